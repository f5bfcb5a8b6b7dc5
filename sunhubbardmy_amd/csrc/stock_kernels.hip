// stock_kernels.hip -- the submatrix-LR update of the projective sweep (src/dqmc_config_v/
// dqmc_proj_update_submatrix_LR.f90, src/dqmc_config_u/dqmc_proj_update_submatrix_LR.f90): the fields of a stock
// of up to 64 sites are decided on F = UR_P (UL UR)^-1 UL_P, then (UL UR)^-1 takes their product.
//   kp_stock_pre    R = UR_P (UL UR)^-1 and Utmp = (UL UR)^-1 UL_P, the sites' rows and columns read in place
//   kp_stock_f      F = R UL_P
//   kp_stock_sites, kp_stock_bonds
//                   the decisions: exchange steps on H = 1 - F, which leave T = Gamma^-1 =
//                   (diag(1/delta) + F_PP)^-1 of the accepted sites P; zero rows and columns elsewhere,
//                   so that the products below take the whole stock without a gather
//   kp_stock_vtmp   Vtmp = T R, and UR's accepted rows times 1 + delta
//   kp_stock_flush  (UL UR)^-1 -= Utmp Vtmp
// Bound by latencies: a product's workgroup streams its 32 x 32 tile's operands once from L2, and the decisions are
// a serial chain.  A stock of 64 sites, eight chains of N = 648, ne = 324: 25 + 8 + 35 + 7 + 17 us (39, 18, 10 and
// 19 us for the products in 32 x 32 tiles dealt out without regard to the XCDs).  Before:
// gathers, five products of 57 us each on 64 x 64 tiles and 162 us of decisions bordering Gamma^-1 one
// bond at a time, with the whole F and Gamma^-1 in LDS.
#include "pqmc_kernels.h"

// site s of a stock: nf < 0 the consecutive sites from ib0, else bond ib0 + s/2 of family nf
__device__ __forceinline__ int stock_site(const PChain &c, int nf, int ib0, int s)
{
    if (nf < 0) return ib0 + s;
    return gp(c.bonds)[2 * (nf * c.nn_lf + ib0) + s];
}

// tiles: the 32 x 16 tiles of R, row by row of tiles, then those of Utmp
extern "C" __global__ void __launch_bounds__(256, 2)
kp_stock_pre(const PChain *chains, int nch, int grp, int nf, int ib0, int nup)
{
    const int ne0 = chains[0].ne, rt = (nup - 1) / 32 + 1, te16 = (ne0 - 1) / 16 + 1, te32 = (ne0 - 1) / 32 + 1;
    int ch, tile;
    if (!tile_of(rt * te16 + ((nup - 1) / 16 + 1) * te32, nch, grp, ch, tile)) return;
    const PChain &c = chains[ch];
    const int n = c.n, ne = c.ne, ns = c.ns, l16 = threadIdx.x & 15;
    GAS cplx *UR = gp(c.UR), *UL = gp(c.UL), *I = gp(c.ULRINV);
    if (tile < rt * te16) {
        const int s0 = tile / te16 * 32, t0 = tile % te16 * 16;
        const int sa = stock_site(c, nf, ib0, min(s0 + l16, nup - 1)), sb = stock_site(c, nf, ib0, min(s0 + 16 + l16, nup - 1));
        GAS cplx *R = gp(c.Rrows);
        gemm_small_tile<2, 1>(
            ne, [=](int i, int k) { return gld(UR + ((size_t)(i < 16 ? sa : sb) + (size_t)k * n)); },
            [=](int k, int j) { return gld(I + ((size_t)k + (size_t)min(t0 + j, ne - 1) * ne)); },
            [=](int i, int j, cplx v) {
                if (s0 + i < nup && t0 + j < ne) gst(R + ((size_t)(s0 + i) + (size_t)(t0 + j) * ns), v);
            });
    } else {
        const int q = tile - rt * te16, t0 = q % te32 * 32, s0 = q / te32 * 16;
        const int sa = stock_site(c, nf, ib0, min(s0 + l16, nup - 1));
        GAS cplx *U = gp(c.Utmp);
        gemm_small_tile<2, 1>(
            ne, [=](int i, int k) { return gld(I + ((size_t)min(t0 + i, ne - 1) + (size_t)k * ne)); },
            [=](int k, int j) { return gld(UL + ((size_t)k + (size_t)sa * ne)); },
            [=](int i, int j, cplx v) {
                if (t0 + i < ne && s0 + j < nup) gst(U + ((size_t)(t0 + i) + (size_t)(s0 + j) * ne), v);
            });
    }
}

// 16 x 16 tiles: at 64 x 64 x 324 four times as many as of 32 x 32, each a quarter of the chain of MFMAs
extern "C" __global__ void __launch_bounds__(256, 2)
kp_stock_f(const PChain *chains, int nch, int grp, int nf, int ib0, int nup)
{
    const int nt = (nup - 1) / 16 + 1;
    int ch, tile;
    if (!tile_of(nt * nt, nch, grp, ch, tile)) return;
    const PChain &c = chains[ch];
    const int ne = c.ne, ns = c.ns, l16 = threadIdx.x & 15, tm = tile % nt * 16, tn = tile / nt * 16;
    const int sa = stock_site(c, nf, ib0, min(tn + l16, nup - 1));
    GAS cplx *R = gp(c.Rrows), *UL = gp(c.UL), *F = gp(c.Felms);
    gemm_small_tile<1, 1>(
        ne, [=](int i, int k) { return gld(R + ((size_t)min(tm + i, nup - 1) + (size_t)k * ns)); },
        [=](int k, int j) { return gld(UL + ((size_t)k + (size_t)sa * ne)); },
        [=](int i, int j, cplx v) {
            if (tm + i < nup && tn + j < nup) gst(F + ((size_t)(tm + i) + (size_t)(tn + j) * ns), v);
        });
}

// what the two decision kernels share: H = 1 - F, T into Ginv (zero outside P), the accepted sites and deltas
struct StockBase {
    const PChain &c;
    int ns, nup;
    __device__ __forceinline__ cplx load(int i, int j)
    {
        const cplx f = gld(gp(c.Felms) + ((size_t)i + (size_t)j * ns));
        return make_double2((i == j ? 1.0 : 0.0) - f.x, -f.y);
    }
    __device__ __forceinline__ void store(int i, int j, cplx v, int ri, int rj)
    {
        const bool in = ri >= 0 && rj >= 0;
        gst(gp(c.Ginv) + ((size_t)i + (size_t)j * ns), make_double2(in ? v.x : 0.0, in ? v.y : 0.0));
    }
    __device__ __forceinline__ void done_base(int ka, cplx phase, int per)
    {
        c.ikd[0] = ka;
        c.sc[SC_PHASE] = phase.x;
        c.sc[SC_PHASE + 1] = phase.y;
        c.sc[SC_ACC] += ka / per;
        c.sc[SC_TRIED] += nup / per;
    }
};

struct StockSites : StockBase {
    int32_t *cf;
    const double *u;
    int i0, isp;
    cplx db;
    __device__ __forceinline__ void factors(int s, cplx &d, cplx &qf, double &u2)
    {
        const int lc = c.ulcomp, is = cf[s], fl = (int)ceil(u[2 * s] * (lc - 1));
        isp = (is + fl - 1) % lc + 1;
        const int k = (fl - 1) + (lc - 1) * (is - 1);
        d = db = c.ud[k];
        qf = cscale(c.uratio[k], c.ug[isp - 1] / c.ug[is - 1]);
        u2 = u[2 * s + 1];
    }
    __device__ __forceinline__ void finish(int s, int rank)
    {
        cf[s] = isp;
        c.xvec[rank] = i0 + s;
        c.Dvec[rank] = db;
    }
    __device__ __forceinline__ void done(int ka, cplx phase) { done_base(ka, phase, 1); }
};

template <int NT, int NF>
__global__ void __launch_bounds__(64 * NT, 2)
kp_stock_sites(const PChain *chains, int nt, int i0, int nup, size_t uoff)
{
    const PChain &c = chains[blockIdx.x];
    StockSites p = {{c, c.ns, nup}, c.uconf + (size_t)(nt - 1) * c.n + i0, c.unif + uoff, i0, 1, {}};
    exchange_block<NT, false, false, NF>(p, nup, c.nflr, make_double2(c.sc[SC_PHASE], c.sc[SC_PHASE + 1]));
}

struct StockBonds : StockBase {
    int32_t *cf;
    const double *u;
    int nf, ib0;
    cplx db;
    __device__ __forceinline__ void factors(int s, cplx &d, cplx &qf, double &u2)
    {
        d = db = c.vd[2 * (cf[s >> 1] - 1) + (s & 1)];
        qf = make_double2(1.0, 0.0);
        u2 = u[2 * (s >> 1) + 1];
    }
    __device__ __forceinline__ void finish(int s, int rank)
    {
        c.xvec[rank] = stock_site(c, nf, ib0, s);
        c.Dvec[rank] = db;
        if (!(s & 1)) cf[s >> 1] = 3 - cf[s >> 1];   // iflip = ceiling(u) = 1 for the two-valued field
    }
    __device__ __forceinline__ void done(int ka, cplx phase) { done_base(ka, phase, 2); }
};

template <int NT>
__global__ void __launch_bounds__(64 * NT, 2)
kp_stock_bonds(const PChain *chains, int nt, int nf, int ib0, int nb, int uoff)
{
    const PChain &c = chains[blockIdx.x];
    StockBonds p = {{c, c.ns, 2 * nb}, c.conf + ((size_t)(nt - 1) * c.nn_nf + nf) * c.n + ib0, c.unif + uoff, nf, ib0, {}};
    exchange_block<NT, false, true, 1>(p, 2 * nb, 1, make_double2(c.sc[SC_PHASE], c.sc[SC_PHASE + 1]));
}

// tiles: those of Vtmp, then 32 columns of UR each: UR(x_m, :) += D_m UR(x_m, :)
// (dqmc_proj_update_submatrix_LR.f90:249-254)
extern "C" __global__ void __launch_bounds__(256, 2)
kp_stock_vtmp(const PChain *chains, int nch, int grp, int nup)
{
    const int te = (chains[0].ne - 1) / GS + 1, rt = (nup - 1) / GS + 1;
    int ch, tile;
    if (!tile_of(te * (rt + 1), nch, grp, ch, tile)) return;
    const PChain &c = chains[ch];
    const int n = c.n, ne = c.ne, ns = c.ns, t0 = tile % te * GS, s0 = tile / te * GS;
    if (tile >= te * rt) {
        const int ik = c.ikd[0];
        GAS cplx *UR = gp(c.UR);
        for (int e = threadIdx.x; e < ik * GS; e += 256) {
            const int m = e % ik, l = t0 + e / ik;
            if (l < ne) {
                GAS cplx *p = UR + ((size_t)c.xvec[m] + (size_t)l * n);
                const cplx v = gld(p), dv = c.Dvec[m];
                gst(p, cadd(v, cmul(dv, v)));
            }
        }
        return;
    }
    GAS cplx *T = gp(c.Ginv), *R = gp(c.Rrows), *V = gp(c.Vtmp);
    gemm_small_tile<2, 2>(
        nup, [=](int i, int k) { return gld(T + ((size_t)min(s0 + i, nup - 1) + (size_t)k * ns)); },
        [=](int k, int j) { return gld(R + ((size_t)k + (size_t)min(t0 + j, ne - 1) * ns)); },
        [=](int i, int j, cplx v) {
            if (s0 + i < nup && t0 + j < ne) gst(V + ((size_t)(s0 + i) + (size_t)(t0 + j) * ns), v);
        });
}

extern "C" __global__ void __launch_bounds__(256, 2)
kp_stock_flush(const PChain *chains, int nch, int grp, int nup)
{
    const int te = (chains[0].ne - 1) / GS + 1;
    int ch, tile;
    if (!tile_of(te * te, nch, grp, ch, tile)) return;
    const PChain &c = chains[ch];
    const int ne = c.ne;
    zgemm_small<0, 0>(c.Utmp, ne, c.Vtmp, c.ns, c.ULRINV, ne, ne, ne, nup, tile % te * GS, tile / te * GS, -1.0, 0.0, 1.0, 0.0);
}

#define STOCK(NT)                                                                              \
    template __global__ void kp_stock_sites<NT, 0>(const PChain *, int, int, int, size_t);      \
    template __global__ void kp_stock_sites<NT, 2>(const PChain *, int, int, int, size_t);      \
    template __global__ void kp_stock_bonds<NT>(const PChain *, int, int, int, int, int);
STOCK(1)
STOCK(2)
STOCK(3)
STOCK(4)
