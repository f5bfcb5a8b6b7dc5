// update_kernels.hip -- the local update of the on-site HS field of one slice, for every form of
// the reference's update (src/dqmc_config_u/dqmc_update.f90, dqmc_update_delay.f90:39-128,
// dqmc_update_submatrix.f90:55-162: the three take the same decisions and differ in how much of G
// they keep current).
//
// The sites are visited in blocks of UB = 64 consecutive sites.  The decisions of a block read
// only the 64 x 64 diagonal block of G, so three kernels take turns per block:
//   k_upd_sites   one workgroup per chain: the block's sequential decisions, with the block of G in
//                 registers and brought up to date after every accepted site;
//   k_upd_panel   64-row strips of every chain: A = G(:, P) T and V = (G(P, :) - E_P) of the ka
//                 accepted sites P;
//   k_upd_flush   64 x 64 tiles of every chain: G += A V, rank ka, on FP64 MFMA.
// With W = diag(1/delta_p) + 1 - G(P, P) and T = W^-1 the product of the accepted single-site
// updates is G + G(:, P) T (G(P, :) - E_P).  T needs no factorization of its own: the sites kernel
// runs Gauss-Jordan exchange steps (below) that leave it in the rows and columns of P.
//
// Why this split: keeping the delayed vectors of all N rows next to the decisions costs a pass over
// N k entries per site in one workgroup (2 us per site at N = 256, k = 32) and a rank-k update of G
// on one CU; here a decision touches 64 x 64 entries and every flop of O(N^2) runs on the whole
// chip.  Per slice: one N = 288 chain 1.72 -> 0.31 ms, 72 chains of N = 64, 144, 256 0.90 -> 0.33 ms,
// 256 chains of N = 256 1.20 -> 1.03 ms (per block 52 us of decisions, 59 us of panels, 148 us of
// flush; one read and write of the 256 MiB of G takes 111 us), 16 chains of N = 64 172 -> 43 us, one
// N = 16 chain 51 -> 8.8 us.
#include "sunhip_kernels.h"

#define UB 64

// the factors of one site's draw that do not depend on G
struct UpdSite {
    cplx db, qf;    // delta(iflip, is), gaml(isp)/gaml(is) phase_ratio(iflip, is)
    double u2;      // the acceptance uniform
    int isp;
};

// The decisions of sites s0 .. s0 + nb - 1, nb <= 16 Q.  Thread (ti, tj) of the 16 x 16 workgroup
// holds the entries (ti + 16 a, tj + 16 b), a, b < Q, of the block H.  Per site: one barrier, after
// which every thread evaluates the same decision from the published diagonal entry, the accepted
// site's column and row come from LDS (published by their owners at the end of the previous site,
// double-buffered, so that one barrier orders both directions) and H takes a rank-1 update.
// WHOLE (the block is all of G, n <= 64): H is G and the update is the plain
//   G += sigma G(:, s) (G(s, :) - e_s), sigma = delta / (1 + delta (1 - G(s, s))),
// written back at the end.  Otherwise H starts as the block of G and takes the exchange step
//   H_ij += sigma H_is H_sj,  H_is = sigma H_is,  H_sj = sigma H_sj,  H_ss = sigma   (i, j != s):
// rows and columns outside P then hold the current G, and H(P, P) = T.
// Bound by the serial chain of one decision (barrier, LDS round trip, the complex products of the
// ratio, one reciprocal) and, for an accepted site, Q^2 complex FMAs per thread.
// Acceptance is |Re(ratiotot phase)| > u2 |Re(phase)| with ratiotot = ratio1^nflr qf: the
// reference's |Re(ratiotot phase) / Re(phase)| > u2 without the division, which lets phase grow
// unnormalised over the block.
template <int Q, bool WHOLE>
__global__ void __launch_bounds__(256)
k_upd_sites(const DChain *chains, int nt, int slice_in_pass, int s0)
{
    __shared__ cplx colb[2][UB], rowb[2][UB];
    __shared__ UpdSite sf[UB + 1];
    const DChain &c = chains[blockIdx.x];
    const int n = c.n;
    if (s0 >= n) return;
    const int nb = min(16 * Q, n - s0);
    const int t = threadIdx.x, ti = t & 15, tj = t >> 4;
    GAS cplx *G = gp(c.G) + ((size_t)s0 + (size_t)s0 * n);
    cplx h[Q][Q];
#pragma unroll
    for (int b = 0; b < Q; b++)
#pragma unroll
        for (int a = 0; a < Q; a++) {
            const int i = ti + 16 * a, j = tj + 16 * b;
            const cplx g = gld(G + ((size_t)min(i, nb - 1) + (size_t)min(j, nb - 1) * n));
            h[a][b] = i < nb && j < nb ? g : make_double2(0.0, 0.0);
        }
    int32_t *cf = c.conf + (size_t)(nt - 1) * n + s0;
    if (t < nb) {
        const double *u = c.unif + (size_t)2 * n * slice_in_pass + 2 * (s0 + t);
        const int is = cf[t], fl = (int)ceil(u[0] * (c.lcomp - 1)), isp = (is + fl - 1) % c.lcomp + 1;
        const int k = (fl - 1) + (c.lcomp - 1) * (is - 1);
        UpdSite q;
        q.db = c.delta_bmat[k];
        q.qf = cscale(c.phase_ratio[k], c.gaml[isp - 1] / c.gaml[is - 1]);
        q.u2 = u[1];
        q.isp = isp;
        sf[t] = q;
    }
    const int nflr = c.nflr;
    cplx phase = make_double2(c.sc[SC_PHASE], c.sc[SC_PHASE + 1]);
    unsigned long long mask = 0;
    int p = 0;
    auto publish = [&](int l, int x, int buf) {
        if (tj == l)
#pragma unroll
            for (int a = 0; a < Q; a++) colb[buf][ti + 16 * a] = h[a][x];
        if (ti == l)
#pragma unroll
            for (int b = 0; b < Q; b++) rowb[buf][tj + 16 * b] = h[x][b];
    };
    publish(0, 0, 0);
#pragma unroll
    for (int x = 0; x < Q; x++) {
        for (int l = 0; l < 16; l++) {
            const int s = 16 * x + l;
            if (s >= nb) break;
            __syncthreads();
            const UpdSite q = sf[s];
            const cplx g = colb[p][s];
            cplx cv[Q], rv[Q];
#pragma unroll
            for (int a = 0; a < Q; a++) cv[a] = colb[p][ti + 16 * a];
#pragma unroll
            for (int b = 0; b < Q; b++) rv[b] = rowb[p][tj + 16 * b];
            const cplx r1 = cadd(cmul(make_double2(1.0 - g.x, -g.y), q.db), make_double2(1.0, 0.0));
            cplx rt = cmul(r1, q.qf);
            for (int f = 1; f < nflr; f++) rt = cmul(rt, r1);
            const cplx ph = cmul(rt, phase);
            const double rd = 1.0 / cabs2(r1);
            // every thread evaluates the same decision; lane 0's makes the branch scalar
            if (__builtin_amdgcn_readfirstlane((int)(fabs(ph.x) > q.u2 * fabs(phase.x))) != 0) {
                const cplx sg = cscale(cmul(q.db, cconj(r1)), rd);
                phase = ph;
                mask |= 1ull << s;
                if (WHOLE) {
                    if (tj == l) rv[x].x -= 1.0;
                } else {
                    if (ti == l) {
                        cv[x] = make_double2(1.0, 0.0);
#pragma unroll
                        for (int b = 0; b < Q; b++) h[x][b] = make_double2(0.0, 0.0);
                    }
                    if (tj == l) {
                        rv[x] = make_double2(1.0, 0.0);
#pragma unroll
                        for (int a = 0; a < Q; a++) h[a][x] = make_double2(0.0, 0.0);
                    }
                }
#pragma unroll
                for (int a = 0; a < Q; a++) {
                    const cplx v = cmul(cv[a], sg);
#pragma unroll
                    for (int b = 0; b < Q; b++) {
                        h[a][b].x += v.x * rv[b].x - v.y * rv[b].y;
                        h[a][b].y += v.x * rv[b].y + v.y * rv[b].x;
                    }
                }
            }
            p ^= 1;
            if (l < 15)
                publish(l + 1, x, p);
            else if (x + 1 < Q)
                publish(0, x + 1, p);
        }
    }
    const int ka = __popcll(mask);
    auto rank = [&](int i) { return __popcll(mask & ((1ull << i) - 1)); };
    if (WHOLE) {
#pragma unroll
        for (int b = 0; b < Q; b++)
#pragma unroll
            for (int a = 0; a < Q; a++) {
                const int i = ti + 16 * a, j = tj + 16 * b;
                if (i < nb && j < nb) gst(G + ((size_t)i + (size_t)j * n), h[a][b]);
            }
    } else {
        GAS cplx *T = gp(c.updt);
#pragma unroll
        for (int b = 0; b < Q; b++)
#pragma unroll
            for (int a = 0; a < Q; a++) {
                const int i = ti + 16 * a, j = tj + 16 * b;
                if ((mask >> i & 1) && (mask >> j & 1)) gst(T + (rank(i) + UB * rank(j)), h[a][b]);
            }
        if (t < nb && (mask >> t & 1)) c.updp[1 + rank(t)] = s0 + t;
        if (t == 0) c.updp[0] = ka;
    }
    if (t < nb && (mask >> t & 1)) cf[t] = sf[t].isp;
    if (t == 0) {
        phase = cscale(phase, 1.0 / sqrt(cabs2(phase)));
        c.sc[SC_PHASE] = phase.x;
        c.sc[SC_PHASE + 1] = phase.y;
        c.sc[SC_ACC] += ka;
        c.sc[SC_TRIED] += nb;
    }
}

// acc += la(i, k) lb(k, j) over k < kk on one 64 x 64 tile, the MFMA layout and LDS staging of
// zgemm_tile; la and lb return zero outside the operands.  K chunks of 16, the next chunk's
// operands in registers while the current one's MFMAs run.
template <class LA, class LB>
__device__ __forceinline__ void mma64(int kk, LA la, LB lb, double4_t (&accr)[2][2], double4_t (&acci)[2][2])
{
    __shared__ double sAr[GT][GK + 1], sAi[GT][GK + 1];
    __shared__ double sBr[GK][GT + 1], sBi[GK][GT + 1];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, wm = w & 1, wn = w >> 1, l16 = lane & 15;
    cplx va[4], vb[4];
    auto load_k = [&](int k0) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int idx = t + 256 * q;
            va[q] = la(idx % GT, k0 + idx / GT);
            vb[q] = lb(k0 + idx % GK, idx / GK);
        }
    };
    load_k(0);
    for (int k0 = 0; k0 < kk; k0 += GK) {
        if (k0 > 0) __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int idx = t + 256 * q, i = idx % GT, k = idx / GT, k2 = idx % GK, j = idx / GK;
            sAr[i][k] = va[q].x; sAi[i][k] = va[q].y;
            sBr[k2][j] = vb[q].x; sBi[k2][j] = vb[q].y;
        }
        __syncthreads();
        if (k0 + GK < kk) load_k(k0 + GK);
        const int ke = min(GK, kk - k0);
#pragma unroll
        for (int ks = 0; ks < GK / 4; ks++) {
            if (4 * ks >= ke) break;
            const int k = 4 * ks + (lane >> 4);
            double xr[2], xi[2], yr[2], yi[2];
#pragma unroll
            for (int s = 0; s < 2; s++) {
                xr[s] = sBr[k][32 * wn + 16 * s + l16]; xi[s] = sBi[k][32 * wn + 16 * s + l16];
                yr[s] = sAr[32 * wm + 16 * s + l16][k]; yi[s] = sAi[32 * wm + 16 * s + l16][k];
            }
#pragma unroll
            for (int sn = 0; sn < 2; sn++)
#pragma unroll
                for (int sm = 0; sm < 2; sm++) {
                    accr[sm][sn] = mfma(xr[sn], yr[sm], accr[sm][sn]);
                    accr[sm][sn] = mfma(-xi[sn], yi[sm], accr[sm][sn]);
                    acci[sm][sn] = mfma(xr[sn], yi[sm], acci[sm][sn]);
                    acci[sm][sn] = mfma(xi[sn], yr[sm], acci[sm][sn]);
                }
        }
    }
}

// rows i0 .. i0 + 63 of A = G(:, P) T (into avec, leading dimension n) and columns i0 .. i0 + 63 of
// V = G(P, :) - E_P (into bvec, column j at 64 j).  P lies within 64 consecutive rows, so the row
// gather reads whole 1 KiB runs; a wave takes a column at a time, lane m the row P[m].
extern "C" __global__ void __launch_bounds__(256)
k_upd_panel(const DChain *chains, int s0)
{
    __shared__ int P[UB];
    const DChain &c = chains[blockIdx.z];
    const int n = c.n, i0 = blockIdx.x * GT;
    if (s0 >= n || i0 >= n) return;
    const int ka = c.updp[0];
    if (ka <= 0) return;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    if (t < UB) P[t] = c.updp[1 + min(t, ka - 1)];
    __syncthreads();
    GAS cplx *G = gp(c.G), *V = gp(c.bvec), *A = gp(c.avec), *T = gp(c.updt);
    {
        const int pm = P[lane];
        for (int q0 = 0; q0 < 16; q0 += 8) {
            cplx v[8];
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] = gld(G + ((size_t)pm + (size_t)min(i0 + 4 * (q0 + q) + w, n - 1) * n));
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int j = i0 + 4 * (q0 + q) + w;
                if (pm == j) v[q].x -= 1.0;
                if (lane < ka && j < n) gst(V + ((size_t)j * UB + lane), v[q]);
            }
        }
    }
    double4_t accr[2][2] = {}, acci[2][2] = {};
    mma64(ka,
          [=](int i, int k) {
              const cplx g = gld(G + ((size_t)min(i0 + i, n - 1) + (size_t)P[min(k, UB - 1)] * n));
              return k < ka ? g : make_double2(0.0, 0.0);
          },
          [=](int k, int j) {
              const cplx g = gld(T + (min(k, ka - 1) + UB * min(j, ka - 1)));
              return k < ka && j < ka ? g : make_double2(0.0, 0.0);
          },
          accr, acci);
    const int wm = w & 1, wn = w >> 1;
#pragma unroll
    for (int sm = 0; sm < 2; sm++)
#pragma unroll
        for (int sn = 0; sn < 2; sn++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = i0 + 32 * wm + 16 * sm + (lane & 15), col = 32 * wn + 16 * sn + (lane >> 4) + 4 * r;
                if (row < n && col < ka) gst(A + ((size_t)row + (size_t)col * n), make_double2(accr[sm][sn][r], acci[sm][sn][r]));
            }
}

// G += A V over 64 x 64 tiles, the accumulators loaded with the tile of G while the first chunk of
// A and V is on its way.  The tiles of a chain are dealt to one XCD (workgroups go round the eight
// XCDs in launch order), whose L2 then holds the chain's A and V: nch8 = the chain count rounded
// up to 8, nt = tiles per side of the largest chain.
extern "C" __global__ void __launch_bounds__(256)
k_upd_flush(const DChain *chains, int nch, int nt, int s0)
{
    const int g = blockIdx.x / (8 * nt * nt), q = blockIdx.x % (8 * nt * nt);
    const int ch = g * 8 + (q & 7), tile = q >> 3;
    if (ch >= nch) return;
    const DChain &c = chains[ch];
    const int n = c.n, i0 = tile % nt * GT, j0 = tile / nt * GT;
    if (s0 >= n || i0 >= n || j0 >= n) return;
    const int ka = c.updp[0];
    if (ka <= 0) return;
    GAS cplx *G = gp(c.G), *V = gp(c.bvec), *A = gp(c.avec);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wm = w & 1, wn = w >> 1;
    double4_t accr[2][2], acci[2][2];
#pragma unroll
    for (int sm = 0; sm < 2; sm++)
#pragma unroll
        for (int sn = 0; sn < 2; sn++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = min(i0 + 32 * wm + 16 * sm + (lane & 15), n - 1);
                const int col = min(j0 + 32 * wn + 16 * sn + (lane >> 4) + 4 * r, n - 1);
                const cplx v = gld_nt(G + ((size_t)row + (size_t)col * n));
                accr[sm][sn][r] = v.x;
                acci[sm][sn][r] = v.y;
            }
    mma64(ka,
          [=](int i, int k) {
              const cplx a = gld(A + ((size_t)min(i0 + i, n - 1) + (size_t)min(k, ka - 1) * n));
              return k < ka ? a : make_double2(0.0, 0.0);
          },
          [=](int k, int j) {
              const cplx b = gld(V + ((size_t)min(j0 + j, n - 1) * UB + min(k, ka - 1)));
              return k < ka ? b : make_double2(0.0, 0.0);
          },
          accr, acci);
#pragma unroll
    for (int sm = 0; sm < 2; sm++)
#pragma unroll
        for (int sn = 0; sn < 2; sn++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = i0 + 32 * wm + 16 * sm + (lane & 15), col = j0 + 32 * wn + 16 * sn + (lane >> 4) + 4 * r;
                if (row < n && col < n)
                    gst_nt(G + ((size_t)row + (size_t)col * n), make_double2(accr[sm][sn][r], acci[sm][sn][r]));
            }
}
