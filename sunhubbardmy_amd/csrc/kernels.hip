// kernels.hip -- CDNA4 (gfx950) kernels of the DQMC sweep.  Every kernel is batched over
// independent Markov chains: blockIdx.z (GEMM, elementwise) or blockIdx.x (one workgroup per
// chain) selects the chain, whose matrix dimension may differ from its neighbours'.
#include "gemm_small.h"

#define FULL_DBL 1

// ------------------------------------------------------------------------------------------
// SFMT19937 on the device (lib/m_spring.f90:187-379): every chain owns its generator; state =
// 624 uint32 lanes + index, kept in global memory between calls.
// ------------------------------------------------------------------------------------------
// Steps i0 .. i0 + L - 1 of the recursion on the 156 words of 128 bits at w (LDS), by one wave of 64:
//   o_i = a_i ^ (a_i << 8) ^ ((b_i >> 11) & mask) ^ (o_{i-2} >> 8) ^ (o_{i-1} << 18)
// (a_i the word's old value, b_i word i + 122 mod 156, the shifts by 8 over 128 bits, the others over 32).  b_i
// is 34 steps back, so for L <= 34 the first three terms of all steps are formed at once by the whole wave;
// the last two run in order in lanes 12 .. 15, one 32-bit part each (lane 15 shifts in zeros from beyond its row).
template <int L>
__device__ __forceinline__ void sfmt_steps(uint32_t *w, int i0, uint32_t &r1, uint32_t &r2)
{
    const int lane = threadIdx.x & 63, l = lane & 3;
    const uint32_t msk = l == 0 ? 0xdfffffefu : l == 1 ? 0xddfecb7fu : l == 2 ? 0xbffaffffu : 0xbffffff6u;
#pragma unroll
    for (int e = lane; e < 4 * L; e += 64) {
        const int i = i0 + (e >> 2), ib = i < 34 ? i + 122 : i - 34;
        const uint32_t a = w[4 * i + l], b = w[4 * ib + l], al = l > 0 ? w[4 * i + l - 1] : 0u;
        w[4 * i + l] = a ^ __builtin_amdgcn_alignbit(a, al, 24) ^ ((b >> 11) & msk);
    }
    __syncthreads();
    if (lane >= 12 && lane < 16) {
        uint32_t t[L];
#pragma unroll
        for (int k = 0; k < L; k++) t[k] = w[4 * (i0 + k) + l];
#pragma unroll
        for (int k = 0; k < L; k++) {
            const uint32_t up = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)r1, 0x101, 0xf, 0xf, true);   // row_shl:1
            const uint32_t o = t[k] ^ __builtin_amdgcn_alignbit(up, r1, 8) ^ (r2 << 18);
            w[4 * (i0 + k) + l] = o;
            r1 = r2;
            r2 = o;
        }
    }
    __syncthreads();
}

__device__ static void sfmt_refill(uint32_t *w)
{
    const int l = threadIdx.x & 3;
    uint32_t r1 = w[4 * 154 + l], r2 = w[4 * 155 + l];
    for (int i0 = 0; i0 < 136; i0 += 34) sfmt_steps<34>(w, i0, r1, r2);
    sfmt_steps<20>(w, 136, r1, r2);
}

// init_gen_rand(seed) and the period certification (lib/m_spring.f90:187-243)
__device__ static void sfmt_seed_state(uint32_t *w, int32_t seed)
{
    const uint32_t parity[4] = {0x00000001u, 0x00000000u, 0x00000000u, 0x13c9e684u};
    w[0] = (uint32_t)seed;
    for (int i = 1; i < 624; i++) w[i] = 1812433253u * (w[i - 1] ^ (w[i - 1] >> 30)) + (uint32_t)i;
    uint32_t inner = 0;
    for (int i = 0; i < 4; i++) inner ^= w[i] & parity[i];
    for (int sh = 16; sh > 0; sh >>= 1) inner ^= inner >> sh;
    if ((inner & 1u) != 1u) {
        bool done = false;
        for (int i = 0; i < 4 && !done; i++) {
            uint32_t work = 1;
            for (int j = 0; j < 32; j++) {
                if (work & parity[i]) { w[i] ^= work; done = true; break; }
                work <<= 1;
            }
        }
    }
    w[624] = 624;
}

extern "C" __global__ void k_sfmt_seed(const DChain *chains, int nchains, const int32_t *seeds)
{
    int ci = blockIdx.x * blockDim.x + threadIdx.x;
    if (ci >= nchains) return;
    sfmt_seed_state(chains[ci].rng, seeds[ci]);
}

// Draws tot numbers from the generator whose state (624 words + index) is at g, one workgroup
// of 64 threads: the state is kept in LDS, and the whole wave converts and stores each block; emit(k, u)
// receives draw k (0-based) of this call.  Bound by the serial part of the recursion: 156 steps of about
// seven dependent instructions a block.  A pass's draws of an N = 288 chain 2.21 -> 0.63 ms, of N = 64 0.31 -> 0.09
// (before, whole steps in one lane, their LDS reads and writes in the chain).
template <typename Emit>
__device__ static void sfmt_draw_block(uint32_t *g, size_t tot, Emit emit)
{
    __shared__ uint32_t w[624];
    for (int i = threadIdx.x; i < 624; i += blockDim.x) w[i] = g[i];
    int idx = (int)g[624];
    __syncthreads();
    size_t k = 0;
    while (k < tot) {
        if (idx >= 624) {
            sfmt_refill(w);
            idx = 0;
        }
        const int cnt = (int)min((size_t)(624 - idx), tot - k);
        for (int j = threadIdx.x; j < cnt; j += blockDim.x)
            emit(k + j, ((double)w[idx + j] + 0.5) * (1.0 / 4294967296.0));
        idx += cnt;
        k += cnt;
        __syncthreads();
    }
    for (int i = threadIdx.x; i < 624; i += blockDim.x) g[i] = w[i];
    if (threadIdx.x == 0) g[624] = (uint32_t)idx;
    __syncthreads();   // a following call in the same workgroup reads the state back
}

// one workgroup per chain; mode 0: fresh HS field conf(i,nt) = ceiling(u*lcomp) (nt outer);
// mode 1: the pass's 2*N*ltrot uniforms
extern "C" __global__ void __launch_bounds__(64)
k_sfmt_draw(const DChain *chains, int nchains, int mode)
{
    const DChain &c = chains[blockIdx.x];
    if (mode == 0) {
        // hconf%input_plqconf, u0conf%input_conf, then v0conf%input_conf (src/dqmc_ft_ctrl.f90:19-35)
        if (c.lwrapp) {
            int32_t *cp = c.confp;
            sfmt_draw_block(c.rng, (size_t)c.lqp * c.ltrot, [=](size_t k, double u) { cp[k] = (int32_t)ceil(u * 4); });
        }
        if (c.lwrapu) {
            const int lc = c.lcomp;
            int32_t *conf = c.conf;
            sfmt_draw_block(c.rng, (size_t)c.n * c.ltrot, [=](size_t k, double u) { conf[k] = (int32_t)ceil(u * lc); });
        }
        if (c.lwrapv) {
            int32_t *cv = c.confv;
            sfmt_draw_block(c.rng, (size_t)c.n * c.nn_nf * c.ltrot, [=](size_t k, double u) { cv[k] = (int32_t)ceil(u * 2); });
        }
    } else if (!c.lwrapv && !c.lwrapp) {
        double *un = c.unif;
        sfmt_draw_block(c.rng, (size_t)2 * c.n * c.ltrot, [=](size_t k, double u) { un[k] = u; });
    } else {
        // per slice the on-site draws (2 n, when the Hubbard field is on), the bond draws
        // (2 nn_nf nn_lf) and the plaquette draws (2 lqp) in the order the pass consumes them:
        // b0 (mode 1) on-site, bonds, plaquettes; 0b (mode 2) plaquettes, bonds, on-site
        // (dqmc_ft_sweep_b0.f90:70-100, dqmc_ft_sweep_0b.f90:82-112)
        double *un = c.unif, *uv = c.unifv, *up = c.unifp;
        const size_t nu = c.lwrapu ? (size_t)2 * c.n : 0, nv = c.lwrapv ? (size_t)2 * c.nn_nf * c.nn_lf : 0;
        const size_t np = c.lwrapp ? (size_t)2 * c.lqp : 0, per = nu + nv + np;
        const bool ufirst = mode == 1;
        sfmt_draw_block(c.rng, per * c.ltrot, [=](size_t k, double u) {
            const size_t s = k / per, r = k % per;
            if (ufirst) {
                if (r < nu) un[s * nu + r] = u;
                else if (r < nu + nv) uv[s * nv + r - nu] = u;
                else up[s * np + r - nu - nv] = u;
            } else {
                if (r < np) up[s * np + r] = u;
                else if (r < np + nv) uv[s * nv + r - np] = u;
                else un[s * nu + r - np - nv] = u;
            }
        });
    }
}

// ------------------------------------------------------------------------------------------
// Kinetic and interaction propagation, checkerboard form (BREAKUP_T).
//   column pass (left products, rows mixed): a workgroup owns CPB full columns in LDS.
//   row pass (right products, columns mixed): a workgroup owns RPB full rows in LDS (ld n + 1).
// Program bits: 1 = families 0..nn_nf-1, 2 = V scaling, 4 = families nn_nf-1..0,
//               8 = V scaling before everything.  Several slices can be chained (B products).
// Bond 2x2 blocks are column-major [T11, T21, T12, T22] (dqmc_left_forward_prop.f90:18-44).
// ------------------------------------------------------------------------------------------
#define CPB 8
#define RPB 8

// one bond per thread (and a stride of columns): the bond's endpoints and 2x2 block are read
// once per family and applied to every column the thread covers
template <class Chain>
__device__ __forceinline__ void cb_left_fams(const Chain &c, cplx *lds, int ncol, const cplx *T, bool rev)
{
    const int nf = c.nn_nf, nl = c.nn_lf, n = c.n;
    const int groups = max(1, (int)blockDim.x / nl);
    const int b = threadIdx.x % nl, g = threadIdx.x / nl;
    for (int q = 0; q < nf; q++) {
        int f = rev ? nf - 1 - q : q;
        for (int bb = b; bb < nl; bb += blockDim.x) {
            if (g >= groups) break;
            const int ist = f * nl + bb;
            const int i1 = c.bonds[2 * ist], i2 = c.bonds[2 * ist + 1];
            const cplx t0 = T[4 * ist], t1 = T[4 * ist + 1], t2 = T[4 * ist + 2], t3 = T[4 * ist + 3];
            for (int cc = g; cc < ncol; cc += groups) {
                cplx x = lds[cc * n + i1], y = lds[cc * n + i2];
                lds[cc * n + i1] = cadd(cmul(t0, x), cmul(t2, y));
                lds[cc * n + i2] = cadd(cmul(t1, x), cmul(t3, y));
            }
        }
        __syncthreads();
    }
}

__device__ static void cb_left_v(const DChain &c, cplx *lds, int ncol, int nt, int vsel)
{
    const int n = c.n;
    GAS const int32_t *cf = gp(c.conf + (size_t)(nt - 1) * n);
    const cplx *vt = vtab_lds(c, vsel);
#pragma unroll 8
    for (int e = threadIdx.x; e < n * ncol; e += blockDim.x) {
        int r = e % n;
        lds[e] = cmul(vt[cf[r] - 1], lds[e]);
    }
    __syncthreads();
}

extern "C" __global__ void __launch_bounds__(256)
k_cb_cols(const DChain *chains, int msel, int pt, int ksel, int prog, int vsel, int nt0, int nt1, int ntstep)
{
    extern __shared__ cplx lds[];
    const DChain &c = chains[blockIdx.z];
    const int n = c.n;
    const int c0 = blockIdx.x * CPB;
    if (c0 >= n) return;
    const int ncol = min(CPB, n - c0);
    cplx *M = chain_mat(c, msel, pt);
    const cplx *T = ksel ? c.ktm1 : c.kt;
    // the CPB columns are one contiguous run of n * ncol elements
    GAS cplx *Mc = gp(M) + (size_t)c0 * n;
    stage_in(lds, n * ncol, [=](int e) { return gld(Mc + (e)); });
    __syncthreads();
    // slices nt0, nt0+ntstep, ..., nt1 (ntstep = +-1); the count bounds the loop
    const int nslice = (ntstep > 0 ? nt1 - nt0 : nt0 - nt1) + 1;
    for (int q = 0, nt = nt0; q < nslice; q++, nt += ntstep) {
        if (nt < 1 || nt > c.ltrot) break;
        if ((prog & 8) && c.lwrapu) cb_left_v(c, lds, ncol, nt, vsel);
        if ((prog & 1) && c.lwrapT) cb_left_fams(c, lds, ncol, T, false);
        if ((prog & 2) && c.lwrapu) cb_left_v(c, lds, ncol, nt, vsel);
        if ((prog & 4) && c.lwrapT) cb_left_fams(c, lds, ncol, T, true);
    }
    stage_out(lds, n * ncol, [=](int e, cplx v) { gst(Mc + (e), v); });
}

// rows in LDS are row-major with the padded leading dimension ldr = n + 1 (lds[rr * ldr + col]):
// the lanes of a family pass touch consecutive sites of one row, and the staging writes of
// eight consecutive rows fall on different banks
__host__ __device__ __forceinline__ int cb_ldr(int n) { return n + 1; }

template <class Chain>
__device__ __forceinline__ void cb_right_fams(const Chain &c, cplx *lds, int nrow, const cplx *T, bool rev)
{
    const int ldr = cb_ldr(c.n);
    const int nf = c.nn_nf, nl = c.nn_lf;
    const int groups = max(1, (int)blockDim.x / nl);
    const int b = threadIdx.x % nl, g = threadIdx.x / nl;
    for (int q = 0; q < nf; q++) {
        int f = rev ? nf - 1 - q : q;
        for (int bb = b; bb < nl; bb += blockDim.x) {
            if (g >= groups) break;
            const int ist = f * nl + bb;
            const int i1 = c.bonds[2 * ist], i2 = c.bonds[2 * ist + 1];
            const cplx t0 = T[4 * ist], t1 = T[4 * ist + 1], t2 = T[4 * ist + 2], t3 = T[4 * ist + 3];
            for (int rr = g; rr < nrow; rr += groups) {
                cplx x = lds[rr * ldr + i1], y = lds[rr * ldr + i2];
                lds[rr * ldr + i1] = cadd(cmul(x, t0), cmul(y, t1));
                lds[rr * ldr + i2] = cadd(cmul(x, t2), cmul(y, t3));
            }
        }
        __syncthreads();
    }
}

__device__ static void cb_right_v(const DChain &c, cplx *lds, int nt, int vsel)
{
    const int n = c.n;
    GAS const int32_t *cf = gp(c.conf + (size_t)(nt - 1) * n);
    const cplx *vt = vtab_lds(c, vsel);
    const int ldr = cb_ldr(n);
#pragma unroll 8
    for (int e = threadIdx.x; e < n * RPB; e += blockDim.x) {
        const int rr = e / n, col = e % n;
        lds[rr * ldr + col] = cmul(lds[rr * ldr + col], vt[cf[col] - 1]);
    }
    __syncthreads();
}

extern "C" __global__ void __launch_bounds__(256)
k_cb_rows(const DChain *chains, int msel, int pt, int ksel, int prog, int vsel, int nt)
{
    extern __shared__ cplx lds[];
    const DChain &c = chains[blockIdx.z];
    const int n = c.n;
    const int r0 = blockIdx.x * RPB;
    if (r0 >= n) return;
    const int nrow = min(RPB, n - r0);
    cplx *M = chain_mat(c, msel, pt);
    const cplx *T = ksel ? c.ktm1 : c.kt;
    // lds[rr * ldr + col] = M(r0 + rr, col): eight consecutive threads read one 128-byte run
    GAS cplx *Mg = gp(M);
    const int ldr = cb_ldr(n);
    stage_in_map<ST_BATCH>(lds, n * RPB, [=](int e) {
        const int rr = e % RPB, col = e / RPB;
        return rr < nrow ? gld(Mg + ((size_t)(r0 + rr) + (size_t)col * n)) : make_double2(0.0, 0.0);
    }, [=](int e) { return (e % RPB) * ldr + e / RPB; });
    __syncthreads();
    if ((prog & 8) && c.lwrapu) cb_right_v(c, lds, nt, vsel);
    if ((prog & 1) && c.lwrapT) cb_right_fams(c, lds, nrow, T, false);
    if ((prog & 2) && c.lwrapu) cb_right_v(c, lds, nt, vsel);
    if ((prog & 4) && c.lwrapT) cb_right_fams(c, lds, nrow, T, true);
    for (int base = threadIdx.x; base < n * RPB; base += ST_BATCH * blockDim.x) {
        cplx v[ST_BATCH];
#pragma unroll
        for (int u = 0; u < ST_BATCH; u++) {
            const int e = base + u * (int)blockDim.x;
            v[u] = e < n * RPB ? lds[(e % RPB) * ldr + e / RPB] : make_double2(0.0, 0.0);
        }
#pragma unroll
        for (int u = 0; u < ST_BATCH; u++) {
            const int e = base + u * (int)blockDim.x, rr = e % RPB, col = e / RPB;
            if (e < n * RPB && rr < nrow) gst(Mg + ((size_t)(r0 + rr) + (size_t)col * n), v[u]);
        }
    }
}

// exp(V) scalings for the dense-K form: rows (side 0) or columns (side 1), or both (side 2:
// rows by vsel, columns by vsel2)
extern "C" __global__ void __launch_bounds__(256)
k_vscale(const DChain *chains, int msel, int pt, int side, int vsel, int vsel2, int nt)
{
    const DChain &c = chains[blockIdx.z];
    const int n = c.n;
    if (!c.lwrapu) return;
    size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)n * n) return;
    int r = (int)(e % n), col = (int)(e / n);
    const int32_t *cf = c.conf + (size_t)(nt - 1) * n;
    cplx *M = chain_mat(c, msel, pt);
    cplx v = M[e];
    if (side == 0 || side == 2) v = cmul(vtab(c, vsel, cf[r]), v);
    if (side == 1) v = cmul(v, vtab(c, vsel, cf[col]));
    if (side == 2) v = cmul(v, vtab(c, vsel2, cf[col]));
    M[e] = v;
}

// ------------------------------------------------------------------------------------------
// Batched ZGEMM on FP64 MFMA (v_mfma_f64_16x16x4_f64), C = alpha op(A) op(B) + beta C,
// all N x N of the chain.  Workgroup tile 64x64, 4 waves of 32x32, K chunk 16 staged in LDS.
// The accumulator holds the transposed tile so that stores are 256-byte column runs.
// MFMA operand layout (probed on gfx950): A(16x4): lane l holds A[l%16][l/16]; B(4x16): lane l
// holds B[l/16][l%16]; D(16x16): lane l, element r holds D[l/16 + 4r][l%16].
// ------------------------------------------------------------------------------------------

// one 64 x 64 tile (tm, tn) of C (m x n, ldc) = alpha op(A) op(B) + beta C, op(A) m x kk,
// op(B) kk x n; op = 0: as stored, 1: conjugate transpose
template <int OPA, int OPB>
__device__ __forceinline__ void zgemm_tile(const cplx *A_, int lda, const cplx *B_, int ldb, cplx *C_, int ldc, int m, int n,
                                  int kk, int tm, int tn, double ar, double ai, double br, double bi)
{
    GAS cplx *A = gp(A_), *B = gp(B_), *C = gp(C_);
    __shared__ double sAr[GT][GK + 1], sAi[GT][GK + 1];
    __shared__ double sBr[GK][GT + 1], sBi[GK][GT + 1];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int wm = w & 1, wn = w >> 1;
    double4_t accr[2][2], acci[2][2];
    for (int i = 0; i < 2; i++)
        for (int j = 0; j < 2; j++)
            for (int r = 0; r < 4; r++) { accr[i][j][r] = 0.0; acci[i][j][r] = 0.0; }
    // the next k block's operands are loaded into registers (clamped, branch-free addresses)
    // while the current block's MFMAs run from LDS
    cplx va[4], vb[4];
    auto load_k = [&](int k0) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int idx = t + 256 * q;
            int i, k, j;
            if (OPA == 0) { i = idx % GT; k = idx / GT; } else { k = idx % GK; i = idx / GK; }
            const int ic = min(tm + i, m - 1), kc = min(k0 + k, kk - 1);
            const cplx a = OPA == 0 ? gld(A + ((size_t)ic + (size_t)kc * lda)) : cconj(gld(A + ((size_t)kc + (size_t)ic * lda)));
            va[q] = (tm + i < m && k0 + k < kk) ? a : make_double2(0.0, 0.0);
            if (OPB == 0) { k = idx % GK; j = idx / GK; } else { j = idx % GT; k = idx / GT; }
            const int jc = min(tn + j, n - 1), kc2 = min(k0 + k, kk - 1);
            const cplx u = OPB == 0 ? gld(B + ((size_t)kc2 + (size_t)jc * ldb)) : cconj(gld(B + ((size_t)jc + (size_t)kc2 * ldb)));
            vb[q] = (tn + j < n && k0 + k < kk) ? u : make_double2(0.0, 0.0);
        }
    };
    load_k(0);
    for (int k0 = 0; k0 < kk; k0 += GK) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int idx = t + 256 * q;
            int i, k, j;
            if (OPA == 0) { i = idx % GT; k = idx / GT; } else { k = idx % GK; i = idx / GK; }
            sAr[i][k] = va[q].x; sAi[i][k] = va[q].y;
            if (OPB == 0) { k = idx % GK; j = idx / GK; } else { j = idx % GT; k = idx / GT; }
            sBr[k][j] = vb[q].x; sBi[k][j] = vb[q].y;
        }
        __syncthreads();
        if (k0 + GK < kk) load_k(k0 + GK);
#pragma unroll
        for (int ks = 0; ks < GK / 4; ks++) {
            const int k = 4 * ks + (lane >> 4), l16 = lane & 15;
            double xr[2], xi[2], yr[2], yi[2];
            for (int s = 0; s < 2; s++) {
                // transposed product: X = op(B)^T rows (output columns), Y = op(A)^T cols (output rows)
                xr[s] = sBr[k][32 * wn + 16 * s + l16]; xi[s] = sBi[k][32 * wn + 16 * s + l16];
                yr[s] = sAr[32 * wm + 16 * s + l16][k]; yi[s] = sAi[32 * wm + 16 * s + l16][k];
            }
            for (int sn = 0; sn < 2; sn++)
                for (int sm = 0; sm < 2; sm++) {
                    accr[sm][sn] = mfma(xr[sn], yr[sm], accr[sm][sn]);
                    accr[sm][sn] = mfma(-xi[sn], yi[sm], accr[sm][sn]);
                    acci[sm][sn] = mfma(xr[sn], yi[sm], acci[sm][sn]);
                    acci[sm][sn] = mfma(xi[sn], yr[sm], acci[sm][sn]);
                }
        }
        __syncthreads();
    }
    const bool zb = (br == 0.0 && bi == 0.0);
    for (int sm = 0; sm < 2; sm++)
        for (int sn = 0; sn < 2; sn++)
            for (int r = 0; r < 4; r++) {
                int row = tm + 32 * wm + 16 * sm + (lane & 15);
                int col = tn + 32 * wn + 16 * sn + (lane >> 4) + 4 * r;
                if (row < m && col < n) {
                    size_t o = (size_t)row + (size_t)col * ldc;
                    double vr = accr[sm][sn][r], vi = acci[sm][sn][r];
                    double outr = ar * vr - ai * vi, outi = ar * vi + ai * vr;
                    if (!zb) { cplx cv = gld(C + (o)); outr += br * cv.x - bi * cv.y; outi += br * cv.y + bi * cv.x; }
                    gst(C + (o), make_double2(outr, outi));
                }
            }
}

// whether a launch takes the 32 x 32 form.  Per flop it is 8 % slower (256 chains of N = 256: 702 against 648 us), so
// it is taken where the rounds of tiles over the 256 CUs give more than that: 16 chains of N = 400 178
// against 241 us (11 rounds of a quarter tile, 4 of a tile), eight 648 x 324 x 648 products 193 against 304
// (8 and 3), one N = 288 chain 18 against 56.
__host__ inline bool gemm_small(int m, int n, int nch)
{
    auto rounds = [=](int t) { return ((long)((m - 1) / t + 1) * ((n - 1) / t + 1) * nch - 1) / 256 + 1; };
    return 13 * rounds(GS) < 48 * rounds(GT);
}

template <int OPA, int OPB>
__global__ void __launch_bounds__(256, 2)
k_zgemm_small(const DChain *chains, int nch, int grp, int nt, int selA, int ptA, int selB, int ptB, int selC, int ptC,
              double ar, double ai, double br, double bi)
{
    int ch, tile;
    if (!tile_of(nt * nt, nch, grp, ch, tile)) return;
    const DChain &c = chains[ch];
    const int n = c.n;
    const int tm = tile % nt * GS, tn = tile / nt * GS;
    if (tm >= n || tn >= n) return;
    zgemm_small<OPA, OPB>(chain_mat(c, selA, ptA), n, chain_mat(c, selB, ptB), n, chain_mat(c, selC, ptC), n, n, n, n,
                          tm, tn, ar, ai, br, bi);
}

template <int OPA, int OPB>
__global__ void __launch_bounds__(256)
k_zgemm(const DChain *chains, int nch, int grp, int nt, int selA, int ptA, int selB, int ptB, int selC, int ptC,
        double ar, double ai, double br, double bi)
{
    int ch, tile;
    if (!tile_of(nt * nt, nch, grp, ch, tile)) return;
    const DChain &c = chains[ch];
    const int n = c.n;
    const int tm = tile % nt * GT, tn = tile / nt * GT;
    if (tm >= n || tn >= n) return;
    zgemm_tile<OPA, OPB>(chain_mat(c, selA, ptA), n, chain_mat(c, selB, ptB), n, chain_mat(c, selC, ptC), n, n, n, n,
                         tm, tn, ar, ai, br, bi);
}

template __global__ void k_zgemm<0, 0>(const DChain *, int, int, int, int, int, int, int, int, int, double, double, double, double);
template __global__ void k_zgemm<1, 0>(const DChain *, int, int, int, int, int, int, int, int, int, double, double, double, double);
template __global__ void k_zgemm<0, 1>(const DChain *, int, int, int, int, int, int, int, int, int, double, double, double, double);

// ------------------------------------------------------------------------------------------
// Equal-time measurement (src/dqmc_measure/equaltime_measure.f90:1-69, zkint :71-114,
// zint_u :116-125, zspsm :283-299 -> Fourier component at the staggering vector).
// One workgroup per chain; the G(i,j) G(j,i) sum is taken over 32x32 tile pairs staged in LDS.
// ------------------------------------------------------------------------------------------
__device__ static double block_sum(double v, double *red)
{
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    __syncthreads();
    if (lane == 0) red[w] = v;
    __syncthreads();
    double s = 0.0;
    for (int i = 0; i < nw; i++) s += red[i];
    return s;
}

// partial sums of S = sum_ij s_i s_j G(i,j) G(j,i) over one 32x32 tile pair (bi <= bj) per
// workgroup, written to rwork[2 tp]
extern "C" __global__ void __launch_bounds__(256)
k_measure_tiles(const DChain *chains)
{
    __shared__ cplx ta[32][33], tb[32][33];
    __shared__ double red[16];
    const DChain &c = chains[blockIdx.z];
    const int n = c.n;
    const int nb = (n + 31) / 32;
    int tp = blockIdx.x;
    if (tp >= nb * (nb + 1) / 2) return;
    int bi = 0;
    while (tp >= nb - bi) { tp -= nb - bi; bi++; }
    const int bj = bi + tp;
    // the eight G entries of a thread (four per tile, 256 threads) and its stag values are loaded
    // in one batch through global-space pointers (clamped addresses), ahead of the LDS stores
    GAS cplx *G = gp(c.G);
    GAS const double *stg = gp(c.stag);
    constexpr int MT_U = 1024 / 256;
    cplx va[MT_U], vb[MT_U];
    double si_[MT_U], sj_[MT_U];
#pragma unroll
    for (int u = 0; u < MT_U; u++) {
        const int e = threadIdx.x + 256 * u, q = e % 32, p = e / 32;
        const int r1 = bi * 32 + q, c1 = bj * 32 + p, r2 = bj * 32 + q, c2 = bi * 32 + p;
        va[u] = gld(G + ((size_t)min(r1, n - 1) + (size_t)min(c1, n - 1) * n));
        vb[u] = gld(G + ((size_t)min(r2, n - 1) + (size_t)min(c2, n - 1) * n));
        si_[u] = stg[min(r1, n - 1)];
        sj_[u] = stg[min(c1, n - 1)];
    }
#pragma unroll
    for (int u = 0; u < MT_U; u++) {
        const int e = threadIdx.x + 256 * u, q = e % 32, p = e / 32;
        const int r1 = bi * 32 + q, c1 = bj * 32 + p, r2 = bj * 32 + q, c2 = bi * 32 + p;
        ta[q][p] = (r1 < n && c1 < n) ? va[u] : make_double2(0.0, 0.0);
        tb[q][p] = (r2 < n && c2 < n) ? vb[u] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    const double wgt = (bi == bj) ? 1.0 : 2.0;
    double ssr = 0.0, ssi = 0.0;
#pragma unroll
    for (int u = 0; u < MT_U; u++) {
        const int e = threadIdx.x + 256 * u, q = e % 32, p = e / 32;
        const int i = bi * 32 + q, j = bj * 32 + p;
        if (i < n && j < n) {
            const cplx pr = cmul(ta[q][p], tb[p][q]);   // G(i,j) G(j,i)
            const double sg = si_[u] * sj_[u] * wgt;
            ssr += sg * pr.x;
            ssi += sg * pr.y;
        }
    }
    ssr = block_sum(ssr, red);
    ssi = block_sum(ssi, red);
    if (threadIdx.x == 0) {
        c.rwork[2 * blockIdx.x] = ssr;
        c.rwork[2 * blockIdx.x + 1] = ssi;
    }
}

// diagonal and bond terms, the tile partials, and the zphi-weighted bin sums; one workgroup per chain
extern "C" __global__ void __launch_bounds__(256)
k_measure(const DChain *chains)
{
    __shared__ double red[16];
    const DChain &c = chains[blockIdx.x];
    const int n = c.n;
    const cplx *G = c.G;
    double zne_r = 0, zne_i = 0, zu_r = 0, zu_i = 0, zk = 0, trr = 0, tri = 0, ssr = 0, ssi = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        cplx g = G[(size_t)i + (size_t)i * n];
        cplx gc = make_double2(1.0 - g.x, -g.y);
        zne_r += gc.x; zne_i += gc.y;
        cplx g2 = cmul(gc, gc);
        zu_r += g2.x; zu_i += g2.y;
        trr += g.x; tri += g.y;
    }
    const int nbond = c.nn_nf * c.nn_lf;
    for (int b = threadIdx.x; b < nbond; b += blockDim.x) {
        int i0 = c.bonds[2 * b], i1 = c.bonds[2 * b + 1];
        // gfc(i0,i1) = delta - gf(i1,i0); kinetic term -2 Re(gfc(i0,i1))
        double gcr = (i0 == i1 ? 1.0 : 0.0) - G[(size_t)i1 + (size_t)i0 * n].x;
        zk += -2.0 * gcr;
    }
    const int nb = (n + 31) / 32, ntp = nb * (nb + 1) / 2;
    for (int t = threadIdx.x; t < ntp; t += blockDim.x) { ssr += c.rwork[2 * t]; ssi += c.rwork[2 * t + 1]; }
    zne_r = block_sum(zne_r, red); zne_i = block_sum(zne_i, red);
    zu_r = block_sum(zu_r, red); zu_i = block_sum(zu_i, red);
    zk = block_sum(zk, red);
    trr = block_sum(trr, red); tri = block_sum(tri, red);
    ssr = block_sum(ssr, red); ssi = block_sum(ssi, red);
    if (threadIdx.x == 0) {
        double *sc = c.sc;
        cplx phase = make_double2(sc[SC_PHASE], sc[SC_PHASE + 1]);
        double sg = phase.x < 0 ? -1.0 : 1.0;
        cplx zphi = cscale(phase, sg / phase.x);
        double fac = 1.0 - 1.0 / (double)(c.nflr * c.nflr);
        cplx ss = cscale(make_double2(trr - ssr, tri - ssi), fac / (double)c.lq);
        cplx v[5];
        v[0] = make_double2(sg, 0.0);
        v[1] = cmul(cscale(make_double2(zne_r, zne_i), 1.0 / (double)c.lq), zphi);
        v[2] = cmul(make_double2(zk * c.kin_weight, 0.0), zphi);
        v[3] = cmul(make_double2(zu_r, zu_i), zphi);
        v[4] = cmul(ss, zphi);
        sc[SC_NOBS] += 1.0;
        for (int k = 0; k < 5; k++) { sc[SC_OBS + 2 * k] += v[k].x; sc[SC_OBS + 2 * k + 1] += v[k].y; }
    }
}

// ------------------------------------------------------------------------------------------
// Householder QR (zgeqp3 / zgeqrf semantics, LAPACK zlarfg reflectors), one workgroup per
// chain, in place on matrix `sel`; tau -> c.tau, jpvt -> c.jpvt (1-based), log det Q -> ldq.
// pivot = 1: column pivoting on downdated partial norms with the tol3z recompute rule.
// ------------------------------------------------------------------------------------------
__device__ static void block_argmax(double v, int idx, double *rv, int *ri, double *outv, int *outi)
{
    // first index of the largest value
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    wave_argmax_dpp(v, idx);
    __syncthreads();
    if (lane == 0) { rv[w] = v; ri[w] = idx; }
    __syncthreads();
    double bv = rv[0];
    int bi = ri[0];
    for (int i = 1; i < nw; i++)
        if (rv[i] > bv || (rv[i] == bv && ri[i] < bi)) { bv = rv[i]; bi = ri[i]; }
    *outv = bv;
    *outi = bi;
}

// One wave's share of rows r0 + lane + 64 q (q < NQ) of a column, loaded with clamped addresses
// in one batch (entries past n are never used).
template <int NQ>
__device__ __forceinline__ void qr_col_load(GAS cplx *col, int r0, int n, int lane, cplx (&x)[NQ])
{
#pragma unroll
    for (int q = 0; q < NQ; q++) x[q] = gld(col + min(r0 + lane + 64 * q, n - 1));
}

// H^H = I - conj(tau) v v^H on one trailing column held in registers (rows i + lane + 64 q), its
// norm downdate as zlaqp2 (the vn1/vn2 recomputation below tol3z)
template <int NQ>
__device__ __forceinline__ void qr_apply_col(GAS cplx *a, const cplx (&x)[NQ], int i, int j, int n, int lane, cplx tc,
                                             const cplx *v, bool pivot, double *vn1, double *vn2, double tol3z)
{
    double sr = 0.0, si = 0.0;
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const int r = i + lane + 64 * q;
        if (r < n) {
            const cplx vv = v[r], aa = x[q];
            sr += vv.x * aa.x + vv.y * aa.y;     // conj(v) a
            si += vv.x * aa.y - vv.y * aa.x;
        }
    }
    sr = wave_sum_dpp(sr);
    si = wave_sum_dpp(si);
    const cplx f = cmul(tc, make_double2(sr, si));
    double nrm2 = 0.0;
    cplx ai_new = make_double2(0.0, 0.0);
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const int r = i + lane + 64 * q;
        if (r < n) {
            const cplx aa = csub(x[q], cmul(v[r], f));
            gst(a + r, aa);
            if (r > i) nrm2 += cabs2(aa);
            else ai_new = aa;   // r == i happens on lane 0 only
        }
    }
    if (pivot) {
        nrm2 = wave_sum_dpp(nrm2);
        if (lane == 0 && vn1[j] != 0.0) {
            double t = sqrt(cabs2(ai_new)) / vn1[j];
            t = 1.0 - t * t;
            if (t < 0.0) t = 0.0;
            double t2 = t * (vn1[j] / vn2[j]) * (vn1[j] / vn2[j]);
            if (t2 <= tol3z) {
                vn1[j] = (i < n - 1) ? sqrt(nrm2) : 0.0;
                vn2[j] = vn1[j];
            } else {
                vn1[j] *= sqrt(t);
            }
        }
    }
}

// Householder QR, column-at-a-time, with column pivoting (pivot = 1, zgeqp3's choice by the
// downdated partial norms) or in the given order (pivot = 0); R above the diagonal, the
// reflectors below, tau to c.tau, log det Q to ldq[out_pt].  The sweeps' form above N = 512.  Every column a
// wave works on is read once into registers (NQ slots of 64 rows).
extern "C" __global__ void __launch_bounds__(1024)
k_qr(const DChain *chains, int sel, int pivot, int out_pt)
{
    extern __shared__ double qrsh[];
    constexpr int NQ = 16;
    const DChain &c = chains[blockIdx.x];
    const int n = c.n;
    double *vn1 = qrsh, *vn2 = qrsh + n;
    cplx *v = (cplx *)(qrsh + 2 * n);          // n
    __shared__ double rv[16];
    __shared__ int ri[16];
    __shared__ cplx s_tau;
    GAS cplx *A = gp(chain_mat(c, sel, 0));
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    // the unpivoted call keeps the prepivot order that k_prepivot left in jpvt
    if (pivot)
        for (int j = threadIdx.x; j < n; j += blockDim.x) c.jpvt[j] = j + 1;
    if (pivot) {
        for (int j = w; j < n; j += nw) {
            cplx x[NQ];
            qr_col_load<NQ>(A + (size_t)j * n, 0, n, lane, x);
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < NQ; q++)
                if (lane + 64 * q < n) s += cabs2(x[q]);
            s = wave_sum_dpp(s);
            if (lane == 0) { vn1[j] = sqrt(s); vn2[j] = vn1[j]; }
        }
    }
    __syncthreads();
    const double tol3z = sqrt(2.220446049250313e-16);
    for (int i = 0; i < n; i++) {
        if (pivot) {
            double bv = -1.0;
            int bi = i;
            for (int j = i + threadIdx.x; j < n; j += blockDim.x) {
                double a = fabs(vn1[j]);
                if (a > bv) { bv = a; bi = j; }
            }
            double mv;
            int p;
            block_argmax(bv, bi, rv, ri, &mv, &p);
            if (p != i) {
                for (int r = threadIdx.x; r < n; r += blockDim.x) {
                    const cplx t = gld(A + ((size_t)r + (size_t)p * n)), u = gld(A + ((size_t)r + (size_t)i * n));
                    gst(A + ((size_t)r + (size_t)p * n), u);
                    gst(A + ((size_t)r + (size_t)i * n), t);
                }
                __syncthreads();
                if (threadIdx.x == 0) {
                    int32_t it = c.jpvt[p]; c.jpvt[p] = c.jpvt[i]; c.jpvt[i] = it;
                    vn1[p] = vn1[i];
                    vn2[p] = vn2[i];
                }
            }
            __syncthreads();
        }
        // reflector of column i (zlarfg), wave 0
        if (w == 0) {
            GAS cplx *col = A + (size_t)i * n;
            cplx x[NQ];
            qr_col_load<NQ>(col, i + 1, n, lane, x);
            const cplx alpha = gld(col + i);
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < NQ; q++)
                if (i + 1 + lane + 64 * q < n) s += cabs2(x[q]);
            s = wave_sum_dpp(s);
            double xnorm = sqrt(s);
            cplx tau = make_double2(0.0, 0.0);
            cplx scal = make_double2(0.0, 0.0);
            double beta = 0.0;
            bool triv = (xnorm == 0.0 && alpha.y == 0.0);
            if (!triv) {
                double nrm = sqrt(alpha.x * alpha.x + alpha.y * alpha.y + s);
                beta = alpha.x >= 0 ? -nrm : nrm;
                tau = make_double2((beta - alpha.x) / beta, -alpha.y / beta);
                scal = cinv(make_double2(alpha.x - beta, alpha.y));
            }
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                const int r = i + 1 + lane + 64 * q;
                if (r < n) {
                    const cplx xs = triv ? x[q] : cmul(x[q], scal);
                    gst(col + r, xs);
                    v[r] = xs;
                }
            }
            if (lane == 0) {
                if (!triv) gst(col + i, make_double2(beta, 0.0));
                v[i] = make_double2(1.0, 0.0);
                s_tau = tau;
                c.tau[i] = tau;
            }
        }
        __syncthreads();
        const cplx tc = cconj(s_tau);
        // apply H^H to the trailing columns, one wave per column (a second register set for the next column would
        // spill at 1024 threads)
        for (int j = i + 1 + w; j < n; j += nw) {
            cplx xa[NQ];
            qr_col_load<NQ>(A + (size_t)j * n, i, n, lane, xa);
            qr_apply_col<NQ>(A + (size_t)j * n, xa, i, j, n, lane, tc, v, pivot, vn1, vn2, tol3z);
        }
        __syncthreads();
    }
    // log det Q, summed by the whole workgroup
    double sr = 0.0, si = 0.0;
    for (int q = threadIdx.x; q < n; q += blockDim.x) {
        const cplx t = gld(gp(c.tau) + q);
        if (t.x != 0.0 || t.y != 0.0) {
            const cplx qq = cdiv(cscale(t, 2.0 * t.x), cmul(t, cconj(t)));
            const cplx l = clog_(make_double2(1.0 - qq.x, -qq.y));
            sr += l.x;
            si += l.y;
        }
    }
    __shared__ double red[16];
    sr = block_sum(sr, red);
    si = block_sum(si, red);
    if (threadIdx.x == 0) c.ldq[out_pt] = make_double2(sr, si);
}

// Q = H_1 ... H_n from the reflectors in matrix `sel` (zung2r), written to chain point U[pt]
// (dest 0) or Us (dest 1)
extern "C" __global__ void __launch_bounds__(1024)
k_formq(const DChain *chains, int sel, int out_pt)
{
    extern __shared__ double qsh[];
    const DChain &c = chains[blockIdx.x];
    const int n = c.n;
    cplx *v = (cplx *)qsh;
    const cplx *A = chain_mat(c, sel, 0);
    cplx *Q = c.U + (size_t)n * n * out_pt;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    for (size_t e = threadIdx.x; e < (size_t)n * n; e += blockDim.x) Q[e] = make_double2(0.0, 0.0);
    __syncthreads();
    for (int i = n - 1; i >= 0; i--) {
        const cplx tau = c.tau[i];
        for (int r = i + threadIdx.x; r < n; r += blockDim.x)
            v[r] = (r == i) ? make_double2(1.0, 0.0) : A[(size_t)r + (size_t)i * n];
        __syncthreads();
        for (int j = i + 1 + w; j < n; j += nw) {
            cplx *q = Q + (size_t)j * n;
            double sr = 0.0, si = 0.0;
            for (int r = i + lane; r < n; r += 64) {
                cplx vv = v[r], qq = q[r];
                sr += vv.x * qq.x + vv.y * qq.y;
                si += vv.x * qq.y - vv.y * qq.x;
            }
            sr = wave_sum_dpp(sr);
            si = wave_sum_dpp(si);
            cplx f = cmul(tau, make_double2(sr, si));
            for (int r = i + lane; r < n; r += 64) q[r] = csub(q[r], cmul(v[r], f));
        }
        __syncthreads();
        for (int r = i + threadIdx.x; r < n; r += blockDim.x) {
            cplx val = (r == i) ? make_double2(1.0 - tau.x, -tau.y)
                                : make_double2(-(tau.x * v[r].x - tau.y * v[r].y), -(tau.x * v[r].y + tau.y * v[r].x));
            Q[(size_t)r + (size_t)i * n] = val;
        }
        __syncthreads();
    }
}

// D = Re diag(R), V = D^-1 triu(R) P^T (first point, column-pivoted QR) -> D[pt], V[pt]
extern "C" __global__ void __launch_bounds__(256)
k_v_from_qrcp(const DChain *chains, int sel, int pt)
{
    const DChain &c = chains[blockIdx.z];
    const int n = c.n;
    size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)n * n) return;
    int i = (int)(e % n), k = (int)(e / n);
    const cplx *R = chain_mat(c, sel, 0);
    double di = R[(size_t)i + (size_t)i * n].x;
    cplx val = (i <= k) ? cscale(R[(size_t)i + (size_t)k * n], 1.0 / di) : make_double2(0.0, 0.0);
    c.V[(size_t)n * n * pt + (size_t)i + (size_t)(c.jpvt[k] - 1) * n] = val;
    if (k == 0) c.D[(size_t)n * pt + i] = di;
}

// prepivot: Btmp = Bd diag(Dprev); columns sorted by decreasing norm (s_zmcpt); the sorted
// matrix goes to W2, the order to jpvt.  One workgroup per chain; a column's place is the count of
// the columns that come before it (equal norms keep their order; s_zmcpt's selection sort exchanges them).
// A wave scales two columns at a time and the copy moves eight entries per thread at a time,
// every batch's loads issued before its first store (clamped addresses).
extern "C" __global__ void __launch_bounds__(1024)
k_prepivot(const DChain *chains, int dpt)
{
    extern __shared__ double psh[];
    const DChain &c = chains[blockIdx.x];
    const int n = c.n;
    double *vn = psh;
    int *jp = (int *)(psh + n);
    const double *Dp = c.D + (size_t)n * dpt;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    GAS cplx *B = gp(c.W1);
    for (int j = w; j < n; j += 2 * nw) {
        const int j2 = j + nw;
        const bool two = j2 < n;
        const double d1 = Dp[j], d2 = Dp[two ? j2 : j];
        GAS cplx *B1 = B + (size_t)j * n, *B2 = B + (size_t)(two ? j2 : j) * n;
        double s1 = 0.0, s2 = 0.0;
        for (int r0 = lane; r0 < n; r0 += 4 * 64) {
            cplx a1[4], a2[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int r = min(r0 + 64 * u, n - 1);
                a1[u] = gld(B1 + r);
                a2[u] = gld(B2 + r);
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int r = r0 + 64 * u;
                if (r < n) {
                    const cplx b1 = cscale(a1[u], d1);
                    gst(B1 + r, b1);
                    s1 += cabs2(b1);
                    if (two) {
                        const cplx b2 = cscale(a2[u], d2);
                        gst(B2 + r, b2);
                        s2 += cabs2(b2);
                    }
                }
            }
        }
        s1 = wave_sum_dpp(s1);
        s2 = wave_sum_dpp(s2);
        if (lane == 0) {
            vn[j] = s1 == s1 ? sqrt(s1) : -1.0;
            if (two) vn[j2] = s2 == s2 ? sqrt(s2) : -1.0;
        }
    }
    __syncthreads();
    // the columns by falling norm, equal norms in their order: every thread counts how many come
    // before its column (a NaN sorts last)
    for (int j = threadIdx.x; j < n; j += blockDim.x) {
        const double vj = vn[j];
        int rank = 0;
        for (int q = 0; q < n; q++) {
            const double v = vn[q];
            rank += v > vj || (v == vj && q < j) ? 1 : 0;
        }
        jp[rank] = j + 1;
    }
    __syncthreads();
    for (int j = threadIdx.x; j < n; j += blockDim.x) c.jpvt[j] = jp[j];
    GAS cplx *W2 = gp(c.W2);
    const int nn = n * n;
    for (int base = threadIdx.x; base < nn; base += 8 * (int)blockDim.x) {
        cplx v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int e = min(base + u * (int)blockDim.x, nn - 1), r = e % n, k = e / n;
            v[u] = gld(B + ((size_t)r + (size_t)(jp[k] - 1) * n));
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int e = base + u * (int)blockDim.x;
            if (e < nn) gst(W2 + e, v[u]);
        }
    }
}

// after the prepivoted QR of W2: D[pt] = Re diag R, W3 = D^-1 triu(R), W4 = P^T V[vpt]
extern "C" __global__ void __launch_bounds__(256)
k_after_qr(const DChain *chains, int pt, int vsel, int vpt)
{
    const DChain &c = chains[blockIdx.z];
    const int n = c.n;
    size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)n * n) return;
    int i = (int)(e % n), j = (int)(e / n);
    // every load (the pivot index first, then the row of V it names) is issued before the
    // first store, through global-space pointers
    GAS cplx *R = gp(c.W2), *Vp = gp(chain_mat(c, vsel, vpt));
    const int jp = gp(c.jpvt)[i];
    const double di = gld(R + ((size_t)i + (size_t)i * n)).x;
    const cplx r = gld(R + e);
    const cplx vrow = gld(Vp + ((size_t)(jp - 1) + (size_t)j * n));
    gst(gp(c.W3) + e, (i <= j) ? cscale(r, 1.0 / di) : make_double2(0.0, 0.0));
    gst(gp(c.W4) + e, vrow);
    if (j == 0) gp(c.D)[(size_t)n * pt + i] = di;
}

// ------------------------------------------------------------------------------------------
// green_equaltime / green_equaltimebb pieces (src/dqmc_ft_core/green_equaltime.f90:1-107,
// green_equaltimebb.f90:1-84).  Right point R = (U[ptR], D[ptR], V[ptR]) or the saved point;
// left point likewise.  rsel/lsel: 0 = chain point, 1 = saved copy (Us, Ds, Vs).
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ double dmax_of(double d) { return fabs(d) > 1.0 ? fabs(d) : 1.0; }
__device__ __forceinline__ double dmin_of(double d) { return fabs(d) > 1.0 ? (d >= 0 ? 1.0 : -1.0) : d; }

__device__ __forceinline__ const double *dvec_of(const DChain &c, int saved, int pt)
{
    return saved ? c.Ds : c.D + (size_t)c.n * pt;
}

// M = uu/(drmax dlmax) + vv drmin dlmin into W3 (uu in W1, vv in W2); bb = 1: M = UR^H/drmax + VR drmin
extern "C" __global__ void __launch_bounds__(256)
k_green_m(const DChain *chains, int bb, int rsaved, int rpt, int lsaved, int lpt)
{
    __shared__ cplx tile[32][33];
    const DChain &c = chains[blockIdx.z];
    const int n = c.n;
    const int bx = blockIdx.x % ((n + 31) / 32), by = blockIdx.x / ((n + 31) / 32);
    if (by * 32 >= n) return;
    // every thread's four entries (256 threads, 32 x 32 tile) are loaded in one batch through
    // global-space pointers with clamped addresses, ahead of the stores
    GAS const double *dr = gp(dvec_of(c, rsaved, rpt));
    constexpr int GU = 1024 / 256;
    if (!bb) {
        GAS const double *dl = gp(dvec_of(c, lsaved, lpt));
        GAS cplx *W1 = gp(c.W1), *W2 = gp(c.W2), *W3 = gp(c.W3);
        cplx x1[GU], x2[GU];
        double di[GU], dj[GU];
#pragma unroll
        for (int u = 0; u < GU; u++) {
            const int e = threadIdx.x + 256 * u;
            const int i = min(bx * 32 + (e % 32), n - 1), j = min(by * 32 + (e / 32), n - 1);
            const size_t o = (size_t)i + (size_t)j * n;
            x1[u] = gld(W1 + o);
            x2[u] = gld(W2 + o);
            di[u] = dr[i];
            dj[u] = dl[j];
        }
#pragma unroll
        for (int u = 0; u < GU; u++) {
            const int e = threadIdx.x + 256 * u;
            const int i = bx * 32 + (e % 32), j = by * 32 + (e / 32);
            if (i < n && j < n) {
                const double a = 1.0 / (dmax_of(di[u]) * dmax_of(dj[u]));
                const double b = dmin_of(di[u]) * dmin_of(dj[u]);
                gst(W3 + ((size_t)i + (size_t)j * n), cadd(cscale(x1[u], a), cscale(x2[u], b)));
            }
        }
    } else {
        GAS cplx *ur = gp(rsaved ? c.Us : c.U + (size_t)n * n * rpt);
        GAS cplx *vr = gp(rsaved ? c.Vs : c.V + (size_t)n * n * rpt);
        GAS cplx *W3 = gp(c.W3);
        // tile of UR^H: element (i, j) = conj(UR(j, i)); read UR block (by, bx) coalesced
        cplx xu[GU], xv[GU];
        double di[GU];
#pragma unroll
        for (int u = 0; u < GU; u++) {
            const int e = threadIdx.x + 256 * u, q = e % 32, p = e / 32;
            const int r = min(by * 32 + q, n - 1), cc = min(bx * 32 + p, n - 1);
            xu[u] = gld(ur + ((size_t)r + (size_t)cc * n));
            const int i = min(bx * 32 + q, n - 1), j = min(by * 32 + p, n - 1);
            xv[u] = gld(vr + ((size_t)i + (size_t)j * n));
            di[u] = dr[i];
        }
#pragma unroll
        for (int u = 0; u < GU; u++) {
            const int e = threadIdx.x + 256 * u, q = e % 32, p = e / 32;
            const int r = by * 32 + q, cc = bx * 32 + p;
            tile[q][p] = (r < n && cc < n) ? xu[u] : make_double2(0.0, 0.0);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < GU; u++) {
            const int e = threadIdx.x + 256 * u, q = e % 32, p = e / 32;
            const int i = bx * 32 + q, j = by * 32 + p;
            if (i < n && j < n) {
                const cplx uh = cconj(tile[p][q]);
                gst(W3 + ((size_t)i + (size_t)j * n), cadd(cscale(uh, 1.0 / dmax_of(di[u])), cscale(xv[u], dmin_of(di[u]))));
            }
        }
    }
}

// right-hand side X = DRmax^-1 UR^H into W4 (tiled transpose)
extern "C" __global__ void __launch_bounds__(256)
k_green_rhs(const DChain *chains, int rsaved, int rpt)
{
    __shared__ cplx tile[32][33];
    const DChain &c = chains[blockIdx.z];
    const int n = c.n;
    const int nb = (n + 31) / 32;
    const int bx = blockIdx.x % nb, by = blockIdx.x / nb;
    if (by >= nb) return;
    // the thread's four entries and scale factors in one batch (global-space pointers, clamped
    // addresses), ahead of the LDS stores
    GAS const double *dr = gp(dvec_of(c, rsaved, rpt));
    GAS cplx *ur = gp(rsaved ? c.Us : c.U + (size_t)n * n * rpt);
    GAS cplx *W4 = gp(c.W4);
    constexpr int GU = 1024 / 256;
    cplx xu[GU];
    double di[GU];
#pragma unroll
    for (int u = 0; u < GU; u++) {
        const int e = threadIdx.x + 256 * u, q = e % 32, p = e / 32;
        xu[u] = gld(ur + ((size_t)min(by * 32 + q, n - 1) + (size_t)min(bx * 32 + p, n - 1) * n));
        di[u] = dr[min(bx * 32 + q, n - 1)];
    }
#pragma unroll
    for (int u = 0; u < GU; u++) {
        const int e = threadIdx.x + 256 * u, q = e % 32, p = e / 32;
        const int r = by * 32 + q, cc = bx * 32 + p;
        tile[q][p] = (r < n && cc < n) ? xu[u] : make_double2(0.0, 0.0);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < GU; u++) {
        const int e = threadIdx.x + 256 * u, q = e % 32, p = e / 32;
        const int i = bx * 32 + q, j = by * 32 + p;
        if (i < n && j < n) gst(W4 + ((size_t)i + (size_t)j * n), cscale(cconj(tile[p][q]), 1.0 / dmax_of(di[u])));
    }
}

// W1 = UL diag(1/dlmax)
extern "C" __global__ void __launch_bounds__(256)
k_green_ulscale(const DChain *chains, int lsaved, int lpt)
{
    const DChain &c = chains[blockIdx.z];
    const int n = c.n;
    size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)n * n) return;
    int j = (int)(e / n);
    const double *dl = dvec_of(c, lsaved, lpt);
    const cplx *ul = lsaved ? c.Us : c.U + (size_t)n * n * lpt;
    c.W1[e] = cscale(ul[e], 1.0 / dmax_of(dl[j]));
}

// LU with partial pivoting (zgetrf, pivot = largest |Re|+|Im|) of W3 in place, one workgroup per
// chain; log det with the imaginary part folded into (-pi, pi] (s_inv_logdet_lu_z) -> SC_ZLD
extern "C" __global__ void __launch_bounds__(1024)
k_lu(const DChain *chains)
{
    extern __shared__ cplx lsh[];
    const DChain &c = chains[blockIdx.x];
    const int n = c.n;
    cplx *lcol = lsh;           // n
    cplx *lrow = lsh + n;       // n
    __shared__ double rv[16];
    __shared__ int ri[16];
    __shared__ int s_piv;
    __shared__ int s_info;
    cplx *A = c.W3;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    if (threadIdx.x == 0) s_info = 0;
    {
        double bv = -1.0;
        int bi = 0;
        for (int r = threadIdx.x; r < n; r += blockDim.x) {
            cplx a = A[r];
            double v = fabs(a.x) + fabs(a.y);
            if (v > bv) { bv = v; bi = r; }
        }
        double mv;
        int p;
        block_argmax(bv, bi, rv, ri, &mv, &p);
        if (threadIdx.x == 0) s_piv = p;
        __syncthreads();
    }
    for (int k = 0; k < n; k++) {
        const int p = s_piv;
        if (threadIdx.x == 0) c.piv[k] = p;
        if (p != k)
            for (int j = threadIdx.x; j < n; j += blockDim.x) {
                cplx t = A[(size_t)p + (size_t)j * n];
                A[(size_t)p + (size_t)j * n] = A[(size_t)k + (size_t)j * n];
                A[(size_t)k + (size_t)j * n] = t;
            }
        __syncthreads();
        cplx akk = A[(size_t)k + (size_t)k * n];
        bool zero = (akk.x == 0.0 && akk.y == 0.0);
        if (zero && threadIdx.x == 0 && s_info == 0) s_info = k + 1;
        cplx pinv = zero ? make_double2(0.0, 0.0) : cinv(akk);
        for (int r = k + 1 + threadIdx.x; r < n; r += blockDim.x) {
            cplx l = zero ? A[(size_t)r + (size_t)k * n] : cmul(A[(size_t)r + (size_t)k * n], pinv);
            A[(size_t)r + (size_t)k * n] = l;
            lcol[r] = l;
        }
        for (int j = k + 1 + threadIdx.x; j < n; j += blockDim.x) lrow[j] = A[(size_t)k + (size_t)j * n];
        __syncthreads();
        double bv = -1.0;
        int bi = k + 1;
        for (int j = k + 1 + w; j < n; j += nw) {
            cplx *a = A + (size_t)j * n;
            cplx f = lrow[j];
            bool track = (j == k + 1);
            for (int r = k + 1 + lane; r < n; r += 64) {
                cplx v = csub(a[r], cmul(lcol[r], f));
                a[r] = v;
                if (track) {
                    double m = fabs(v.x) + fabs(v.y);
                    if (m > bv) { bv = m; bi = r; }
                }
            }
        }
        double mv;
        int np;
        block_argmax(bv, bi, rv, ri, &mv, &np);
        if (threadIdx.x == 0) s_piv = (k + 1 < n) ? np : 0;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        cplx ld = make_double2(0.0, 0.0);
        for (int i = 0; i < n; i++) {
            cplx d = A[(size_t)i + (size_t)i * n];
            if (c.piv[i] != i) d = make_double2(-d.x, -d.y);
            ld = cadd(ld, clog_(d));
        }
        double im = ld.y;
        double k2 = round(im / 2.0 / M_PI);
        ld.y = im - 2.0 * M_PI * k2;
        c.sc[SC_ZLD] = ld.x;
        c.sc[SC_ZLD + 1] = ld.y;
        c.sc[SC_INFO] = (double)s_info;
    }
}

// solve (P L U) Y = X for X = matrix `xsel`, in place; one wave per right-hand-side column,
// the column held in registers (n <= 1024)
#define SOLVE_SLOTS 16
extern "C" __global__ void __launch_bounds__(512)
k_lu_solve(const DChain *chains, int xsel)
{
    const DChain &c = chains[blockIdx.x];
    const int n = c.n;
    const cplx *A = c.W3;
    cplx *X = chain_mat(c, xsel, 0);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int ns = (n + 63) / 64;
    for (int j = w; j < n; j += nw) {
        cplx *x = X + (size_t)j * n;
        cplx reg[SOLVE_SLOTS];
#pragma unroll
        for (int s = 0; s < SOLVE_SLOTS; s++) {
            int r = lane + 64 * s;
            reg[s] = (s < ns && r < n) ? x[r] : make_double2(0.0, 0.0);
        }
        // row interchanges, in order
        for (int k = 0; k < n; k++) {
            int p = c.piv[k];
            if (p == k) continue;
            int sk = k >> 6, lk = k & 63, sp = p >> 6, lp = p & 63;
            double kr = 0, ki = 0, pr = 0, pi = 0;
#pragma unroll
            for (int s = 0; s < SOLVE_SLOTS; s++) {
                if (s == sk) { kr = __shfl(reg[s].x, lk, 64); ki = __shfl(reg[s].y, lk, 64); }
                if (s == sp) { pr = __shfl(reg[s].x, lp, 64); pi = __shfl(reg[s].y, lp, 64); }
            }
#pragma unroll
            for (int s = 0; s < SOLVE_SLOTS; s++) {
                if (s == sk && lane == lk) reg[s] = make_double2(pr, pi);
                if (s == sp && lane == lp) reg[s] = make_double2(kr, ki);
            }
        }
        // L y = b (unit lower)
        for (int k = 0; k < n - 1; k++) {
            int sk = k >> 6, lk = k & 63;
            double yr = 0, yi = 0;
#pragma unroll
            for (int s = 0; s < SOLVE_SLOTS; s++)
                if (s == sk) { yr = __shfl(reg[s].x, lk, 64); yi = __shfl(reg[s].y, lk, 64); }
            const cplx yk = make_double2(yr, yi);
            const cplx *lk_col = A + (size_t)k * n;
#pragma unroll
            for (int s = 0; s < SOLVE_SLOTS; s++) {
                int r = lane + 64 * s;
                if (s >= sk && s < ns && r > k && r < n) reg[s] = csub(reg[s], cmul(lk_col[r], yk));
            }
        }
        // U x = y
        for (int k = n - 1; k >= 0; k--) {
            int sk = k >> 6, lk = k & 63;
            cplx ukk = A[(size_t)k + (size_t)k * n];
#pragma unroll
            for (int s = 0; s < SOLVE_SLOTS; s++)
                if (s == sk && lane == lk) reg[s] = cdiv(reg[s], ukk);
            double yr = 0, yi = 0;
#pragma unroll
            for (int s = 0; s < SOLVE_SLOTS; s++)
                if (s == sk) { yr = __shfl(reg[s].x, lk, 64); yi = __shfl(reg[s].y, lk, 64); }
            const cplx yk = make_double2(yr, yi);
            const cplx *uk_col = A + (size_t)k * n;
#pragma unroll
            for (int s = 0; s < SOLVE_SLOTS; s++) {
                int r = lane + 64 * s;
                if (s <= sk && r < k) reg[s] = csub(reg[s], cmul(uk_col[r], yk));
            }
        }
#pragma unroll
        for (int s = 0; s < SOLVE_SLOTS; s++) {
            int r = lane + 64 * s;
            if (s < ns && r < n) x[r] = reg[s];
        }
    }
}

// logweightf scratch: general (bb = 0): -ldql + ldqr + zld + sum log dlmax + sum log drmax;
// bb = 1: ldqr + zld + sum log drmax
extern "C" __global__ void __launch_bounds__(256)
k_green_logw(const DChain *chains, int bb, int rsaved, int rpt, int lsaved, int lpt, int dst_logw)
{
    __shared__ double red[16];
    const DChain &c = chains[blockIdx.x];
    const int n = c.n;
    const double *dr = dvec_of(c, rsaved, rpt);
    const double *dl = bb ? nullptr : dvec_of(c, lsaved, lpt);
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        s += log(dmax_of(dr[i]));
        if (!bb) s += log(dmax_of(dl[i]));
    }
    s = block_sum(s, red);
    if (threadIdx.x == 0) {
        cplx ldqr = rsaved ? make_double2(c.sc[SC_LDQ_SAVE], c.sc[SC_LDQ_SAVE + 1]) : c.ldq[rpt];
        cplx lw = cadd(ldqr, make_double2(c.sc[SC_ZLD] + s, c.sc[SC_ZLD + 1]));
        if (!bb) {
            cplx ldql = lsaved ? make_double2(c.sc[SC_LDQ_SAVE], c.sc[SC_LDQ_SAVE + 1]) : c.ldq[lpt];
            lw = csub(lw, ldql);
        }
        c.sc[dst_logw] = lw.x;
        c.sc[dst_logw + 1] = lw.y;
    }
}

// wrap check and replacement (dqmc_ft_sweep_0b.f90:212-259): max|Gs - G|, set_phase of the
// scratch weight, G <- Gs when the LU succeeded; compare = 0 at sweep start (plain set)
extern "C" __global__ void __launch_bounds__(1024)
k_wrap(const DChain *chains, int compare)
{
    __shared__ double red[16];
    __shared__ double cnt_sh[8][16];
    const DChain &c = chains[blockIdx.x];
    const int n = c.n;
    double *sc = c.sc;
    double mx = 0.0;
    bool nonfinite = false;
    // eight entries of Gs (and G) per thread in flight at a time, clamped addresses; the maximum
    // and the flag do not depend on the order
    GAS cplx *Gsg = gp(c.Gs), *Gg = gp(c.G);
    const int nn = n * n;
    for (int base = threadIdx.x; base < nn; base += 8 * (int)blockDim.x) {
        cplx a[8], b[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int e = min(base + u * (int)blockDim.x, nn - 1);
            a[u] = gld(Gsg + e);
            if (compare) b[u] = gld(Gg + e);
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            if (base + u * (int)blockDim.x >= nn) continue;
            if (!isfinite(a[u].x) || !isfinite(a[u].y)) nonfinite = true;
            if (compare) {
                const double d = hypot(a[u].x - b[u].x, a[u].y - b[u].y);
                if (d > mx) mx = d;
            }
        }
    }
    // max reduction
    for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    if (lane == 0) red[w] = mx;
    __syncthreads();
    mx = 0.0;
    for (int i = 0; i < nw; i++) mx = fmax(mx, red[i]);
    // set_phase: exp(i nflr Im logw) * prod_{i,nt} phase(conf) = exp(i (nflr Im logw + sum cnt_l arg_l))
    // counts 0-3: the on-site field's components; 4-7: the plaquette field's (hconf%phase of
    // every plaquette and slice, set_phase.f90:9-15)
    double cnt[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (c.phase_from_conf && c.lwrapu) {
        const int tot = n * c.ltrot;
        GAS const int32_t *cg = gp(c.conf);
        for (int base = threadIdx.x; base < tot; base += 8 * (int)blockDim.x) {
            int v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = cg[min(base + u * (int)blockDim.x, tot - 1)];
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (base + u * (int)blockDim.x < tot) {
                    cnt[0] += (v[u] == 1); cnt[1] += (v[u] == 2); cnt[2] += (v[u] == 3); cnt[3] += (v[u] == 4);
                }
        }
    }
    if (c.lwrapp) {
        size_t tot = (size_t)c.lqp * c.ltrot;
        for (size_t e = threadIdx.x; e < tot; e += blockDim.x) {
            int v = c.confp[e];
            cnt[4] += (v == 1); cnt[5] += (v == 2); cnt[6] += (v == 3); cnt[7] += (v == 4);
        }
    }
    for (int l = 0; l < 8; l++) {
        double v = cnt[l];
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if (lane == 0) cnt_sh[l][w] = v;
    }
    int nf_flag = __syncthreads_or(nonfinite ? 1 : 0);
    if (threadIdx.x == 0) {
        double ang = (double)c.nflr * sc[SC_LOGW_TMP + 1];
        for (int l = 0; l < c.lcomp && l < 4; l++) {
            double s = 0.0;
            for (int i = 0; i < nw; i++) s += cnt_sh[l][i];
            ang += s * c.parg[l];
        }
        if (c.lwrapp)
            for (int l = 0; l < 4; l++) {
                double s = 0.0;
                for (int i = 0; i < nw; i++) s += cnt_sh[4 + l][i];
                ang += s * c.pparg[l];
            }
        cplx ph = make_double2(cos(ang), sin(ang));
        int info = (int)sc[SC_INFO];
        if (nf_flag) sc[SC_NONFINITE] = 1.0;
        if (compare) {
            if (mx > sc[SC_MAXWRAP]) sc[SC_MAXWRAP] = mx;
            cplx ph0 = make_double2(sc[SC_PHASE], sc[SC_PHASE + 1]);
            double pd = hypot(ph0.x - ph.x, ph0.y - ph.y);
            if (pd > sc[SC_MAXPH]) sc[SC_MAXPH] = pd;
            sc[SC_NCHK] += 1.0;
            sc[SC_SUMLOG] += log10(mx > 0 ? mx : 1e-300);
        }
        if (info == 0) {
            sc[SC_LOGW] = sc[SC_LOGW_TMP];
            sc[SC_LOGW + 1] = sc[SC_LOGW_TMP + 1];
            sc[SC_PHASE] = ph.x;
            sc[SC_PHASE + 1] = ph.y;
        }
        red[0] = (double)info;
    }
    __syncthreads();
    if ((int)red[0] == 0) {
        for (int base = threadIdx.x; base < nn; base += 8 * (int)blockDim.x) {
            cplx a[8];
#pragma unroll
            for (int u = 0; u < 8; u++) a[u] = gld(Gsg + min(base + u * (int)blockDim.x, nn - 1));
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (base + u * (int)blockDim.x < nn) gst(Gg + base + u * (int)blockDim.x, a[u]);
        }
    }
    __syncthreads();
    int tn = (int)sc[SC_TRACE_N];
    if (c.trace && tn < c.trace_cap) {
        for (size_t e = threadIdx.x; e < (size_t)n * n; e += blockDim.x) c.trace[(size_t)tn * n * n + e] = c.G[e];
        __syncthreads();
        if (threadIdx.x == 0) sc[SC_TRACE_N] = tn + 1;
    }
}

// ------------------------------------------------------------------------------------------
// small utility kernels
// ------------------------------------------------------------------------------------------
// set chain point pt to (I, 1, I, 0)
extern "C" __global__ void __launch_bounds__(256)
k_set_identity(const DChain *chains, int pt)
{
    const DChain &c = chains[blockIdx.z];
    const int n = c.n;
    size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)n * n) return;
    int i = (int)(e % n), j = (int)(e / n);
    cplx v = make_double2(i == j ? 1.0 : 0.0, 0.0);
    c.U[(size_t)n * n * pt + e] = v;
    c.V[(size_t)n * n * pt + e] = v;
    if (j == 0) c.D[(size_t)n * pt + i] = 1.0;
    if (e == 0) c.ldq[pt] = make_double2(0.0, 0.0);
}

// copy between matrices; mode 1 additionally saves D[pt] and ldq[pt] of the chain point
extern "C" __global__ void __launch_bounds__(256)
k_copy(const DChain *chains, int dsel, int dpt, int ssel, int spt)
{
    const DChain &c = chains[blockIdx.z];
    const int n = c.n;
    size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)n * n) return;
    chain_mat(c, dsel, dpt)[e] = chain_mat(c, ssel, spt)[e];
}

// save chain point pt (U, D, V, logdetQ) into (Us, Ds, Vs, SC_LDQ_SAVE)
extern "C" __global__ void __launch_bounds__(256)
k_save_point(const DChain *chains, int pt)
{
    const DChain &c = chains[blockIdx.z];
    const int n = c.n;
    size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)n * n) return;
    c.Us[e] = c.U[(size_t)n * n * pt + e];
    c.Vs[e] = c.V[(size_t)n * n * pt + e];
    if (e < (size_t)n) c.Ds[e] = c.D[(size_t)n * pt + e];
    if (e == 0) { c.sc[SC_LDQ_SAVE] = c.ldq[pt].x; c.sc[SC_LDQ_SAVE + 1] = c.ldq[pt].y; }
}
