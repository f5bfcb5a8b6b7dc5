// pqmc_kernels.hip -- device side of the projective sweep (src/dqmc_proj_core, vconf of
// src/dqmc_config_v): rectangular propagators UR (N x ne) and UL (ne x N), their inverse
// overlap ULRINV = (UL UR)^-1 (ne x ne), the bond-field operators, the submatrix-LR update and
// the QR / LU steps of the stabilization.  Every kernel is batched over chains that share N, ne
// and the stock size; blockIdx.z (elementwise, GEMM) or blockIdx.x (one workgroup per chain)
// selects the chain.
#include "pqmc_kernels.h"

// ---- batched ZGEMM with explicit shapes: C = alpha A B + beta C --------------------------
struct PGemm {
    int sa, pa, sb, pb, sc, pc;
    int m, n, k, lda, ldb, ldc;
    double ar, ai, br, bi;
};

extern "C" __global__ void __launch_bounds__(256)
kp_gemm(const PChain *chains, int nch, int grp, PGemm g)
{
    const int mt = (g.m - 1) / GT + 1, nt = (g.n - 1) / GT + 1;
    int ch, tile;
    if (!tile_of(mt * nt, nch, grp, ch, tile)) return;
    const PChain &c = chains[ch];
    const int tm = tile % mt * GT, tn = tile / mt * GT;
    if (tm >= g.m || tn >= g.n) return;
    zgemm_tile<0, 0>(pmat(c, g.sa, g.pa), g.lda, pmat(c, g.sb, g.pb), g.ldb, pmat(c, g.sc, g.pc), g.ldc, g.m, g.n,
                     g.k, tm, tn, g.ar, g.ai, g.br, g.bi);
}

extern "C" __global__ void __launch_bounds__(256, 2)
kp_gemm_small(const PChain *chains, int nch, int grp, PGemm g)
{
    const int mt = (g.m - 1) / GS + 1, nt = (g.n - 1) / GS + 1;
    int ch, tile;
    if (!tile_of(mt * nt, nch, grp, ch, tile)) return;
    const PChain &c = chains[ch];
    const int tm = tile % mt * GS, tn = tile / mt * GS;
    if (tm >= g.m || tn >= g.n) return;
    zgemm_small<0, 0>(pmat(c, g.sa, g.pa), g.lda, pmat(c, g.sb, g.pb), g.ldb, pmat(c, g.sc, g.pc), g.ldc, g.m, g.n,
                      g.k, tm, tn, g.ar, g.ai, g.br, g.bi);
}

// ---- copies -------------------------------------------------------------------------------
// dst[e] = src[e] (or conj) for e < count
extern "C" __global__ void __launch_bounds__(256)
kp_copy(const PChain *chains, int dsel, int dpt, int ssel, int spt, int count, int conj)
{
    const PChain &c = chains[blockIdx.z];
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= count) return;
    cplx v = pmat(c, ssel, spt)[e];
    if (conj) v.y = -v.y;
    pmat(c, dsel, dpt)[e] = v;
}

// dst (cols x rows, ld cols) = src^T (or src^H) of src (rows x cols, ld rows); 32 x 32 tiles
extern "C" __global__ void __launch_bounds__(256)
kp_transpose(const PChain *chains, int dsel, int dpt, int ssel, int spt, int rows, int cols, int conj)
{
    __shared__ cplx t[32][33];
    const PChain &c = chains[blockIdx.z];
    const int tr = (rows + 31) / 32;
    const int r0 = (blockIdx.x % tr) * 32, c0 = (blockIdx.x / tr) * 32;
    if (c0 >= cols) return;
    const cplx *S = pmat(c, ssel, spt);
    cplx *D = pmat(c, dsel, dpt);
    for (int e = threadIdx.x; e < 1024; e += blockDim.x) {
        int i = e % 32, j = e / 32;
        if (r0 + i < rows && c0 + j < cols) t[j][i] = S[(size_t)(r0 + i) + (size_t)(c0 + j) * rows];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 1024; e += blockDim.x) {
        int j = e % 32, i = e / 32;   // D(c0+j, r0+i) = S(r0+i, c0+j)
        if (r0 + i < rows && c0 + j < cols) {
            cplx v = t[j][i];
            if (conj) v.y = -v.y;
            D[(size_t)(c0 + j) + (size_t)(r0 + i) * cols] = v;
        }
    }
}

// M (n x n) += diag(1)
extern "C" __global__ void __launch_bounds__(256)
kp_add_identity(const PChain *chains, int sel)
{
    const PChain &c = chains[blockIdx.z];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= c.n) return;
    cplx *M = pmat(c, sel, 0);
    M[(size_t)i + (size_t)i * c.n].x += 1.0;
}

// ---- propagation: kinetic families and bond-field operators -------------------------------
// One launch applies a short program of operators to UR from the left (blockIdx.y = 0, CPB
// columns of UR in LDS) and to UL from the right (blockIdx.y = 1, RPB rows of UL in LDS).
// op kinds: 0 kinetic families 0..nn_nf-1, 1 kinetic families nn_nf-1..0 (checkerboard
// tables kselL / kselR), 2 bond field of family arg with modes modeL / modeR:
//   left  0: rows <- diag(bp,bm) ut rows    (dqmc_config_v/dqmc_left_forward_prop.f90, nflag 2)
//   left  1: rows <- u rows                 (left_forward nflag 1, left_backward nflag 2)
//   left  2: rows <- u diag(bpi,bmi) rows   (dqmc_left_backward_prop.f90, nflag 1)
//   right 0: cols <- cols u diag(bpi,bmi)   (dqmc_right_backward_prop.f90, nflag 2)
//   right 1: cols <- cols u                 (right_backward nflag 1, right_forward nflag 2)
//   right 2: cols <- cols diag(bp,bm) ut    (dqmc_right_forward_prop.f90, nflag 1)
// u = ut = [[1, 1], [1, -1]] / sqrt(2) (src/dqmc_config_v.f90:19-20).
// kind 3: the on-site field, UR rows / UL columns times bmat (mode 0) or bmat_inv (mode 1) of
// the site's value (src/dqmc_config_u/dqmc_left_forward_prop.f90:23-32 and its three siblings).
#define POPS_MAX 12
struct POps {
    int nops, nt, kselL, kselR, sides;   // sides: 1 = UR, 2 = UL
    int kind[POPS_MAX], arg[POPS_MAX], modeL[POPS_MAX], modeR[POPS_MAX];
};

#define HADAMARD 0.70710678118654752440

// the eight bond-field factors in registers (uniform loads); t(is, k) selects without memory access
struct BondTab {
    cplx v[8];
    __device__ BondTab(const PChain &c)
    {
        for (int k = 0; k < 8; k++) v[k] = c.vt[k];
    }
    __device__ __forceinline__ cplx operator()(int is, int k) const { return is == 2 ? v[4 + k] : v[k]; }
};

__device__ __forceinline__ void v_left_pair(const BondTab &tb, int is, int mode, cplx &x, cplx &y)
{
    const cplx s = make_double2(HADAMARD, 0.0), ms = make_double2(-HADAMARD, 0.0);
    const cplx t[4] = {tb(is, 0), tb(is, 1), tb(is, 2), tb(is, 3)};
    if (mode == 2) { x = cmul(t[2], x); y = cmul(t[3], y); }
    cplx v1 = cadd(cmul(s, x), cmul(s, y));
    cplx v2 = cadd(cmul(s, x), cmul(ms, y));
    if (mode == 0) { v1 = cmul(t[0], v1); v2 = cmul(t[1], v2); }
    x = v1;
    y = v2;
}

__device__ __forceinline__ void v_right_pair(const BondTab &tb, int is, int mode, cplx &x, cplx &y)
{
    const cplx s = make_double2(HADAMARD, 0.0), ms = make_double2(-HADAMARD, 0.0);
    const cplx t[4] = {tb(is, 0), tb(is, 1), tb(is, 2), tb(is, 3)};
    if (mode == 2) { x = cmul(x, t[0]); y = cmul(y, t[1]); }
    cplx v1 = cadd(cmul(x, s), cmul(y, s));
    cplx v2 = cadd(cmul(x, s), cmul(y, ms));
    if (mode == 0) { v1 = cmul(t[2], v1); v2 = cmul(t[3], v2); }
    x = v1;
    y = v2;
}

extern "C" __global__ void __launch_bounds__(256)
kp_prop(const PChain *chains, POps ops)
{
    extern __shared__ cplx lds[];
    const PChain &c = chains[blockIdx.z];
    const int n = c.n, ne = c.ne, nl = c.nn_lf;
    const int groups = max(1, (int)blockDim.x / nl);
    const int bt = threadIdx.x % nl, g = threadIdx.x / nl;
    if (!(ops.sides & (1 << blockIdx.y))) return;
    const BondTab tb(c);
    if (blockIdx.y == 0) {
        // UR from the left, CPB columns
        const int c0 = blockIdx.x * CPB;
        if (c0 >= ne) return;
        const int ncol = min(CPB, ne - c0);
        cplx *M = c.UR;
        for (int e = threadIdx.x; e < n * ncol; e += blockDim.x) lds[e] = M[(size_t)(e % n) + (size_t)(c0 + e / n) * n];
        __syncthreads();
        for (int o = 0; o < ops.nops; o++) {
            if (ops.kind[o] < 2) {
                if (c.kmode == 0) cb_left_fams(c, lds, ncol, ops.kselL ? c.ktm1 : c.kt, ops.kind[o] == 1);
                continue;
            }
            if (ops.kind[o] == 3) {
                const int32_t *uc = c.uconf + (size_t)(ops.nt - 1) * n;
                for (int i = threadIdx.x; i < n; i += blockDim.x) {
                    const int is = uc[i] - 1;
                    const cplx fct = ops.modeL[o] ? c.ubi[is] : c.ub[is];
                    for (int cc = 0; cc < ncol; cc++) lds[cc * n + i] = cmul(fct, lds[cc * n + i]);
                }
                __syncthreads();
                continue;
            }
            const int f = ops.arg[o], mode = ops.modeL[o];
            const int32_t *cf = c.conf + ((size_t)(ops.nt - 1) * c.nn_nf + f) * n;
            for (int bb = bt; bb < nl; bb += blockDim.x) {
                if (g >= groups) break;
                const int ist = f * nl + bb;
                const int i1 = c.bonds[2 * ist], i2 = c.bonds[2 * ist + 1];
                const int is = cf[bb];
                for (int cc = g; cc < ncol; cc += groups) {
                    cplx x = lds[cc * n + i1], y = lds[cc * n + i2];
                    v_left_pair(tb, is, mode, x, y);
                    lds[cc * n + i1] = x;
                    lds[cc * n + i2] = y;
                }
            }
            __syncthreads();
        }
        for (int e = threadIdx.x; e < n * ncol; e += blockDim.x) M[(size_t)(e % n) + (size_t)(c0 + e / n) * n] = lds[e];
    } else {
        // UL from the right, RPB rows; lds[rr * ldr + col]
        const int r0 = blockIdx.x * RPB;
        if (r0 >= ne) return;
        const int nrow = min(RPB, ne - r0), ldr = cb_ldr(n);
        cplx *M = c.UL;
        for (int e = threadIdx.x; e < n * RPB; e += blockDim.x) {
            int rr = e % RPB, col = e / RPB;
            lds[rr * ldr + col] = (rr < nrow) ? M[(size_t)(r0 + rr) + (size_t)col * ne] : make_double2(0.0, 0.0);
        }
        __syncthreads();
        for (int o = 0; o < ops.nops; o++) {
            if (ops.kind[o] < 2) {
                if (c.kmode == 0) cb_right_fams(c, lds, nrow, ops.kselR ? c.ktm1 : c.kt, ops.kind[o] == 1);
                continue;
            }
            if (ops.kind[o] == 3) {
                const int32_t *uc = c.uconf + (size_t)(ops.nt - 1) * n;
                for (int e = threadIdx.x; e < n * RPB; e += blockDim.x) {
                    const int rr = e / n, col = e % n;
                    const int is = uc[col] - 1;
                    const cplx fct = ops.modeR[o] ? c.ubi[is] : c.ub[is];
                    lds[rr * ldr + col] = cmul(lds[rr * ldr + col], fct);
                }
                __syncthreads();
                continue;
            }
            const int f = ops.arg[o], mode = ops.modeR[o];
            const int32_t *cf = c.conf + ((size_t)(ops.nt - 1) * c.nn_nf + f) * n;
            for (int bb = bt; bb < nl; bb += blockDim.x) {
                if (g >= groups) break;
                const int ist = f * nl + bb;
                const int i1 = c.bonds[2 * ist], i2 = c.bonds[2 * ist + 1];
                const int is = cf[bb];
                for (int rr = g; rr < nrow; rr += groups) {
                    cplx x = lds[rr * ldr + i1], y = lds[rr * ldr + i2];
                    v_right_pair(tb, is, mode, x, y);
                    lds[rr * ldr + i1] = x;
                    lds[rr * ldr + i2] = y;
                }
            }
            __syncthreads();
        }
        for (int e = threadIdx.x; e < n * RPB; e += blockDim.x) {
            int rr = e % RPB, col = e / RPB;
            if (rr < nrow) M[(size_t)(r0 + rr) + (size_t)col * ne] = lds[rr * ldr + col];
        }
    }
}

// ---- stabilization --------------------------------------------------------------------------
// weight bookkeeping after a scratch inverse (z = log det ULR in SC_ZLD):
//   op 0: sweep start  logweightf = logwDV(nst) + z, phase = exp(i nflr Im z)
//   op 1: 0b point n   logwDV(n) = logwDV(n-1) + rlog, logw = logwDV(n) [+ logwDV(n+1)] + z
//   op 2: b0 point n   logwDV(n+1) = [logwDV(n+2) +] rlog, logw = logwDV(n+1) [+ logwDV(n)] + z
//   op 3: 0b pass start logwDV(0) = 0
//   op 4: start point n logwDV(n) = logwDV(n-1) + rlog
// (dqmc_proj_sweep_start_0b.f90:16-38, dqmc_proj_sweep_0b.f90:121-148, dqmc_proj_sweep_b0.f90:113-141)
extern "C" __global__ void kp_weights(const PChain *chains, int nchains, int op, int n, int phasediff)
{
    const int ci = blockIdx.x * blockDim.x + threadIdx.x;
    if (ci >= nchains) return;
    const PChain &c = chains[ci];
    double *sc = c.sc, *lw = c.logwDV;
    const cplx z = make_double2(sc[SC_ZLD], sc[SC_ZLD + 1]);
    double dv = 0.0;
    if (op == 3) { lw[0] = 0.0; return; }
    if (op == 4) { lw[n] = lw[n - 1] + sc[SC_RLOG]; return; }
    if (op == 0) {
        dv = lw[c.nst];
    } else if (op == 1) {
        lw[n] = lw[n - 1] + sc[SC_RLOG];
        dv = (n == c.nst) ? lw[n] : lw[n] + lw[n + 1];
    } else {
        lw[n + 1] = (n + 1 == c.nst) ? sc[SC_RLOG] : lw[n + 2] + sc[SC_RLOG];
        dv = (n == 0) ? lw[n + 1] : lw[n + 1] + lw[n];
    }
    const cplx logw = make_double2(dv + z.x, z.y);
    // set_phase: exp(i nflr Im logw) times the on-site field's phases (angle sum from kp_uphase)
    const double a = (double)c.nflr * logw.y + ((c.lwrapu && c.uphase_from_conf) ? sc[PS_UANG] : 0.0);
    const cplx ph = make_double2(cos(a), sin(a));
    if (phasediff) {
        const cplx old = make_double2(sc[SC_PHASE], sc[SC_PHASE + 1]);
        const double d = sqrt(cabs2(csub(old, ph)));
        if (d > sc[SC_MAXPH]) sc[SC_MAXPH] = d;
    }
    sc[SC_PHASE] = ph.x;
    sc[SC_PHASE + 1] = ph.y;
    sc[SC_LOGW] = logw.x;
    sc[SC_LOGW + 1] = logw.y;
    if (!(isfinite(logw.x) && isfinite(logw.y))) sc[SC_NONFINITE] = 1.0;
}

// wrap check: max |G2 - G| (s_compare_max_z), one workgroup per chain; the log10 sum and the
// count as the reference's WRAPERROR block; optionally G joins the trace
extern "C" __global__ void __launch_bounds__(256)
kp_wrap_check(const PChain *chains, int compare, int trace)
{
    __shared__ double red[4];
    const PChain &c = chains[blockIdx.x];
    const size_t nn = (size_t)c.n * c.n;
    if (compare) {
        double mx = 0.0;
        for (size_t e = threadIdx.x; e < nn; e += blockDim.x) {
            double d = sqrt(cabs2(csub(c.G2[e], c.G[e])));
            if (!(d <= mx)) mx = d;   // NaN propagates
        }
        for (int o = 32; o > 0; o >>= 1) {
            double v = __shfl_xor(mx, o, 64);
            if (!(v <= mx)) mx = v;
        }
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
        __syncthreads();
        if (threadIdx.x == 0) {
            double m = red[0];
            for (int w = 1; w < (int)(blockDim.x >> 6); w++) if (!(red[w] <= m)) m = red[w];
            if (!isfinite(m)) c.sc[SC_NONFINITE] = 1.0;
            if (m > c.sc[SC_MAXWRAP]) c.sc[SC_MAXWRAP] = m;
            c.sc[SC_NCHK] += 1.0;
            c.sc[SC_SUMLOG] += log10(m > 0.0 ? m : 1e-300);
        }
    }
    if (trace && c.trace) {
        const int k = (int)c.sc[SC_TRACE_N];
        if (k < c.trace_cap) {
            for (size_t e = threadIdx.x; e < nn; e += blockDim.x) c.trace[(size_t)k * nn + e] = c.G[e];
            __syncthreads();
            if (threadIdx.x == 0) c.sc[SC_TRACE_N] = k + 1;
        }
    }
}

// sum over the on-site field of the arguments of phase(conf) into sc[PS_UANG] (set_phase,
// src/dqmc_proj_core/set_phase.f90:16-22); one workgroup per chain
extern "C" __global__ void __launch_bounds__(256)
kp_uphase(const PChain *chains)
{
    const PChain &c = chains[blockIdx.x];
    __shared__ double red[4];
    double a = 0.0;
    if (c.lwrapu)
        for (size_t k = threadIdx.x; k < (size_t)c.n * c.ltrot; k += blockDim.x) a += c.upa[c.uconf[k] - 1];
    a = wave_sum(a);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
    __syncthreads();
    if (threadIdx.x == 0) c.sc[PS_UANG] = (red[0] + red[1]) + (red[2] + red[3]);
}

// draws of the projective chain: mode 0 the fresh fields (the on-site field first, N ltrot
// draws conf(i,nt) = ceiling(u lcomp) with i inner, as u0conf%input_conf precedes
// v0conf%input_conf in dqmc_start; then the bond field, N nn_nf ltrot draws, conf(i,nf,nt)
// with nf innermost), mode 1 the pass's uniforms (per slice 2 N for the on-site field and
// 2 nn_lf nn_nf for the bonds), mode 2 count uniforms of chain `which` into out
extern "C" __global__ void __launch_bounds__(64)
kp_draw(const PChain *chains, int mode, int which, int count, double *out)
{
    const int ci = (mode == 2) ? which : (int)blockIdx.x;
    const PChain &c = chains[ci];
    if (mode == 0) {
        const int n = c.n, nf = c.nn_nf;
        if (c.lwrapu) {
            int32_t *uc = c.uconf;
            const int lc = c.ulcomp;
            sfmt_draw_block(c.rng, (size_t)n * c.ltrot, [=](size_t k, double u) { uc[k] = (int32_t)ceil(u * lc); });
        }
        if (c.lwrapv) {
            int32_t *conf = c.conf;
            sfmt_draw_block(c.rng, (size_t)n * nf * c.ltrot, [=](size_t k, double u) {
                const size_t f = k % nf, i = (k / nf) % n, t = k / ((size_t)nf * n);
                conf[(t * nf + f) * n + i] = (int32_t)ceil(u * 2.0);
            });
        }
    } else if (mode == 1) {
        double *un = c.unif;
        sfmt_draw_block(c.rng, p_slice_draws(c) * c.ltrot, [=](size_t k, double u) { un[k] = u; });
    } else {
        sfmt_draw_block(c.rng, (size_t)count, [=](size_t k, double u) { out[k] = u; });
    }
}

extern "C" __global__ void kp_seed(const PChain *chains, int nchains, const int32_t *seeds)
{
    const int ci = blockIdx.x * blockDim.x + threadIdx.x;
    if (ci >= nchains) return;
    sfmt_seed_state(chains[ci].rng, seeds[ci]);
}


// ------------------------------------------------------------------------------------------
// The G-based updates of the on-site field (src/dqmc_config_u/dqmc_proj_update_delay.f90,
// dqmc_proj_update_submatrix_G.f90): the finite-temperature delay / submatrix kernels run on
// G = 1 - UR (UL UR)^-1 UL through the chain's view; then the rows of UR whose site flipped are
// multiplied by bmat(new) / bmat(old) = 1 + delta_bmat(iflip, old) (urrecord of the reference).
// ------------------------------------------------------------------------------------------
extern "C" __global__ void __launch_bounds__(256)
kp_u_save(const PChain *chains, int nt)
{
    const PChain &c = chains[blockIdx.z];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < c.n) c.uold[i] = c.uconf[(size_t)(nt - 1) * c.n + i];
}

extern "C" __global__ void __launch_bounds__(256)
kp_u_rescale(const PChain *chains, int nt)
{
    const PChain &c = chains[blockIdx.z];
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)c.n * c.ne) return;
    const int i = (int)(e % c.n), lc = c.ulcomp;
    const int old = c.uold[i], nw = c.uconf[(size_t)(nt - 1) * c.n + i];
    if (old == nw) return;
    const int iflip = ((nw - old) % lc + lc) % lc;           // nw = mod(old + iflip - 1, lc) + 1
    const cplx d = c.ud[(iflip - 1) + (lc - 1) * (old - 1)];
    c.UR[e] = cmul(c.UR[e], make_double2(1.0 + d.x, d.y));
}

// the bond field of family nf at slice nt before a G-based update, and UR's rows i1, i2 of every
// bond it flipped times 1 + delta_bmat_p, 1 + delta_bmat_m of the old value
// (src/dqmc_config_v/dqmc_proj_update_delay.f90:124-125; UR is in the family's rotated basis)
extern "C" __global__ void __launch_bounds__(256)
kp_v_save(const PChain *chains, int nt, int nf)
{
    const PChain &c = chains[blockIdx.z];
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < c.nn_lf) c.uold[q] = c.conf[((size_t)(nt - 1) * c.nn_nf + nf) * c.n + q];
}

extern "C" __global__ void __launch_bounds__(256)
kp_v_rescale(const PChain *chains, int nt, int nf)
{
    const PChain &c = chains[blockIdx.z];
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)c.nn_lf * c.ne) return;
    const int q = (int)(e % c.nn_lf), j = (int)(e / c.nn_lf);
    const int old = c.uold[q], nw = c.conf[((size_t)(nt - 1) * c.nn_nf + nf) * c.n + q];
    if (old == nw) return;
    const int ist = nf * c.nn_lf + q;
    const int i1 = c.bonds[2 * ist], i2 = c.bonds[2 * ist + 1];
    const cplx dp = c.vd[2 * (old - 1)], dm = c.vd[2 * (old - 1) + 1];
    cplx *a = c.UR + (size_t)j * c.n;
    a[i1] = cmul(a[i1], make_double2(1.0 + dp.x, dp.y));
    a[i2] = cmul(a[i2], make_double2(1.0 + dm.x, dm.y));
}
