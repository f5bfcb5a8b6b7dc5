// update_kernels.hip -- the local update of the on-site HS field of one slice, for every form of
// the reference's update (src/dqmc_config_u/dqmc_update.f90, dqmc_update_delay.f90:39-128,
// dqmc_update_submatrix.f90:55-162: the three take the same decisions and differ in how much of G
// they keep current).
//
// The sites are visited in blocks of UB = 64 consecutive sites.  The decisions of a block read
// only the 64 x 64 diagonal block of G, so three kernels take turns per block:
//   k_upd_sites   one workgroup per chain: the block's sequential decisions, with the block of G in
//                 registers and brought up to date after every four sites;
//   k_upd_panel   64-row strips of every chain: A = G(:, P) T and V = (G(P, :) - E_P) of the ka
//                 accepted sites P;
//   k_upd_flush   64 x 64 tiles of every chain: G += A V, rank ka, on FP64 MFMA.
// With W = diag(1/delta_p) + 1 - G(P, P) and T = W^-1 the product of the accepted single-site
// updates is G + G(:, P) T (G(P, :) - E_P).  T needs no factorization of its own: the sites kernel
// runs Gauss-Jordan exchange steps (exchange.h) that leave it in the rows and columns of P.
//
// Why this split: keeping the delayed vectors of all N rows next to the decisions costs a pass over
// N k entries per site in one workgroup (2 us per site at N = 256, k = 32) and a rank-k update of G
// on one CU; here a decision touches 64 x 64 entries and every flop of O(N^2) runs on the whole
// chip.  Per slice: one N = 288 chain 1.72 -> 0.23 ms, 72 chains of N = 64, 144, 256 0.90 -> 0.27 ms,
// 256 chains of N = 256 1.20 -> 0.95 ms (per block 40 us of decisions, 55 us of panels, 140 us of
// flush; one read and write of the 256 MiB of G takes 111 us), 16 chains of N = 64 172 -> 31 us.
#include "gemm_small.h"
#include "update_kernels.h"

// the decisions of sites s0 .. of one chain on G; WHOLE: n <= 64 and s0 = 0
template <bool WHOLE>
struct GSites {
    const DChain &c;
    GAS cplx *G;
    int32_t *cf;
    const double *u;
    int n, s0, nb, isp;
    __device__ __forceinline__ cplx load(int i, int j) { return gld(G + ((size_t)i + (size_t)j * n)); }
    __device__ __forceinline__ void factors(int s, cplx &db, cplx &qf, double &u2)
    {
        const int is = cf[s], fl = (int)ceil(u[2 * s] * (c.lcomp - 1));
        isp = (is + fl - 1) % c.lcomp + 1;
        const int k = (fl - 1) + (c.lcomp - 1) * (is - 1);
        db = c.delta_bmat[k];
        qf = cscale(c.phase_ratio[k], c.gaml[isp - 1] / c.gaml[is - 1]);
        u2 = u[2 * s + 1];
    }
    __device__ __forceinline__ void store(int i, int j, cplx v, int ri, int rj)
    {
        if (WHOLE)
            gst(G + ((size_t)i + (size_t)j * n), v);
        else if (ri >= 0 && rj >= 0)
            gst(gp(c.updt) + (ri + UB * rj), v);
    }
    __device__ __forceinline__ void finish(int s, int rank)
    {
        cf[s] = isp;
        if (!WHOLE) c.updp[1 + rank] = s0 + s;
    }
    __device__ __forceinline__ void done(int ka, cplx phase)
    {
        if (!WHOLE) c.updp[0] = ka;
        c.sc[SC_PHASE] = phase.x;
        c.sc[SC_PHASE + 1] = phase.y;
        c.sc[SC_ACC] += ka;
        c.sc[SC_TRIED] += nb;
    }
};

template <int NT, bool WHOLE, int NF>
__global__ void __launch_bounds__(64 * NT, 2)
k_upd_sites(const DChain *chains, int nt, int slice_in_pass, int s0)
{
    const DChain &c = chains[blockIdx.x];
    const int n = c.n;
    if (s0 >= n) return;
    GSites<WHOLE> p = {c, gp(c.G) + ((size_t)s0 + (size_t)s0 * n), c.conf + (size_t)(nt - 1) * n + s0,
                       c.unif + (size_t)2 * n * slice_in_pass + 2 * s0, n, s0, min(16 * NT, n - s0), 1};
    exchange_block<NT, WHOLE, false, NF>(p, p.nb, c.nflr, make_double2(c.sc[SC_PHASE], c.sc[SC_PHASE + 1]));
}

#if !UPD_WHOLE && UPD_NF == 0
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
// V = G(P, :) - E_P (into bvec, column j at 64 j).  A wave takes a column at a time, lane m the row P[m]
// (of the on-site field: within one run of 64 rows).
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
// XCDs in launch order, the chains are taken eight at a time), whose L2 then holds the chain's A and V.
// nt = tiles per side of the largest chain.
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

// The same two products on 32 x 32 tiles with K split over the waves, where those need fewer rounds of the CUs: a
// 64 x 64 x 64 tile is 8 us of one CU's MFMAs, whatever else is idle.  One N = 288 chain: panel 13.8 -> 7.1 us,
// flush 11.7 -> 6.5; 16 of N = 72 12.1 -> 6.3 and 9.7 -> 6.2; 16 of N = 400 the panel 16 -> 9.5.
// A workgroup of the panel forms a tile of A, its share (half of the tile's 32 columns) of V on the way.
extern "C" __global__ void __launch_bounds__(256, 2)
k_upd_panel_small(const DChain *chains, int nch, int grp, int nt, int s0)
{
    __shared__ int P[UB];
    int ch, tile;
    if (!tile_of(2 * nt, nch, grp, ch, tile)) return;
    const DChain &c = chains[ch];
    const int n = c.n, i0 = (tile >> 1) * GS, h = tile & 1;
    if (s0 >= n || i0 >= n) return;
    const int ka = c.updp[0];
    if (ka <= 0) return;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    if (t < UB) P[t] = c.updp[1 + min(t, ka - 1)];
    __syncthreads();
    GAS cplx *G = gp(c.G), *V = gp(c.bvec), *A = gp(c.avec), *T = gp(c.updt);
    const int pm = P[lane], j0 = i0 + 16 * h + w;
    cplx v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = gld(G + ((size_t)pm + (size_t)min(j0 + 4 * q, n - 1) * n));
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int j = j0 + 4 * q;
        if (pm == j) v[q].x -= 1.0;
        if (lane < ka && j < n) gst(V + ((size_t)j * UB + lane), v[q]);
    }
    if (GS * h >= ka) return;
    gemm_small_tile<2, 2>(
        ka, [=](int i, int k) { return gld(G + ((size_t)min(i0 + i, n - 1) + (size_t)P[k] * n)); },
        [=](int k, int j) { return gld(T + (k + UB * min(GS * h + j, ka - 1))); },
        [=](int i, int j, cplx a) {
            if (i0 + i < n && GS * h + j < ka) gst(A + ((size_t)(i0 + i) + (size_t)(GS * h + j) * n), a);
        });
}

extern "C" __global__ void __launch_bounds__(256, 2)
k_upd_flush_small(const DChain *chains, int nch, int grp, int nt, int s0)
{
    int ch, tile;
    if (!tile_of(nt * nt, nch, grp, ch, tile)) return;
    const DChain &c = chains[ch];
    const int n = c.n, i0 = tile % nt * GS, j0 = tile / nt * GS;
    if (s0 >= n || i0 >= n || j0 >= n) return;
    const int ka = c.updp[0];
    if (ka <= 0) return;
    zgemm_small<0, 0>(c.avec, n, c.bvec, UB, c.G, n, n, n, ka, i0, j0, 1.0, 0.0, 1.0, 0.0);
}

// The t-V bond field's decisions of one family (src/dqmc_config_v/dqmc_update.f90, dqmc_update_delay.f90:
// 28-128, dqmc_update_submatrix.f90:63-250: the same decisions), 32 bonds at a time on the block of G at
// their 64 sites, gathered; T and the sites go to k_upd_panel and k_upd_flush as the on-site field's do.
// (The reference's v3(2,1) at dqmc_update_submatrix.f90:153 is -v5(2,1) v5(2,2) / (v5(1,1) det v5), not
// the inverse's -v5(2,1) / det v5; the inverse is used here, with which its three forms agree.)
// 16 chains of N = 72 and 36 bonds a family: 240 us in one workgroup with delayed vectors, 85 us
// here with the panels and the flush (64 x 64 tiles; 67 with the small ones).
struct GBonds {
    const DChain &c;
    GAS cplx *G;
    GAS const int32_t *site;
    int32_t *cf;
    const double *u;
    int n, nb;
    __device__ __forceinline__ cplx load(int i, int j) { return gld(G + ((size_t)site[i] + (size_t)site[j] * n)); }
    __device__ __forceinline__ int flipped(int q) { return (cf[q] - 1 + (int)ceil(u[2 * q])) & 1; }
    __device__ __forceinline__ void factors(int s, cplx &db, cplx &qf, double &u2)
    {
        const int q = s >> 1;
        db = c.vdl[2 * (cf[q] - 1) + (s & 1)];
        qf = make_double2(1.0, 0.0);
        u2 = u[2 * q + 1];
    }
    __device__ __forceinline__ void store(int i, int j, cplx v, int ri, int rj)
    {
        if (ri >= 0 && rj >= 0) gst(gp(c.updt) + (ri + UB * rj), v);
    }
    __device__ __forceinline__ void finish(int s, int rank)
    {
        c.updp[1 + rank] = site[s];
        if (!(s & 1)) cf[s >> 1] = flipped(s >> 1) + 1;
    }
    __device__ __forceinline__ void done(int ka, cplx phase)
    {
        c.updp[0] = ka;
        c.sc[SC_PHASE] = phase.x;
        c.sc[SC_PHASE + 1] = phase.y;
        c.vacc[0] += ka / 2;
        c.vacc[1] += nb / 2;
    }
};

template <int NT>
__global__ void __launch_bounds__(64 * NT, 2)
k_upd_bonds(const DChain *chains, int nt, int nf, int slice, int p, int ib0, int per)
{
    const DChain &c = chains[blockIdx.x];
    const int nl = c.nn_lf;
    if (!c.lwrapv || ib0 >= nl) {
        if (threadIdx.x == 0) c.updp[0] = 0;
        return;
    }
    GBonds b = {c, gp(c.G), gp(c.bonds) + 2 * (nf * nl + ib0), c.confv + ((size_t)(nt - 1) * c.nn_nf + nf) * c.n + ib0,
                c.unifv + (size_t)2 * nl * (c.nn_nf * slice + p) + 2 * ib0, c.n, 2 * min(per, nl - ib0)};
    exchange_block<NT, false, true, 1>(b, b.nb, 1, make_double2(c.sc[SC_PHASE], c.sc[SC_PHASE + 1]));
}
template __global__ void k_upd_bonds<1>(const DChain *, int, int, int, int, int, int);
template __global__ void k_upd_bonds<2>(const DChain *, int, int, int, int, int, int);
template __global__ void k_upd_bonds<3>(const DChain *, int, int, int, int, int, int);
template __global__ void k_upd_bonds<4>(const DChain *, int, int, int, int, int, int);
#endif

// one object file per (WHOLE, NF) pair, so that they compile side by side
template __global__ void k_upd_sites<1, UPD_WHOLE, UPD_NF>(const DChain *, int, int, int);
template __global__ void k_upd_sites<2, UPD_WHOLE, UPD_NF>(const DChain *, int, int, int);
template __global__ void k_upd_sites<3, UPD_WHOLE, UPD_NF>(const DChain *, int, int, int);
template __global__ void k_upd_sites<4, UPD_WHOLE, UPD_NF>(const DChain *, int, int, int);
