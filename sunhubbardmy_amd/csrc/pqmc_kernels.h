// pqmc_kernels.h -- the projective chain's descriptor and the kernels of stock_kernels.hip, a translation
// unit of its own.
#pragma once
#include "exchange.h"
#include "factor.h"
#include "gemm_small.h"

// scalar slots of the projective chain beyond the shared layout (SC_PHASE, SC_LOGW, SC_ZLD,
// SC_INFO, SC_OBS ... keep their meaning)
// (the projective sweep has no saved chain point, so SC_LDQ_SAVE's first slot holds the angle
// sum of the on-site field's phases)
enum { PS_UANG = SC_LDQ_SAVE };

enum {
    P_UR = 0, P_UL, P_ULRINV, P_ULR, P_T1, P_T2, P_ULO, P_URO, P_INV2, P_G, P_G2, P_KT, P_KTM1,
    P_UST, P_PROJ
};

struct PChain {
    int n, ne, nn_nf, nn_lf, kmode, ns, ltrot, nst, nflr, lq, trace_cap;
    cplx *UR, *UL, *ULRINV, *ULR, *T1, *T2, *ULo, *URo, *INV2, *G, *G2, *Ust, *proj;
    cplx *Rrows, *Felms, *Ginv, *Vtmp, *Utmp, *Dvec;
    cplx *tau, *tblk, *trace;
    int32_t *piv, *conf, *xvec, *ikd;
    double *unif, *sc, *logwDV, *rwork;
    uint32_t *rng;
    const int32_t *bonds;
    const cplx *kt, *ktm1;
    const double *stag;
    cplx vt[8];   // (bp, bm, bpi, bmi) for field value 1 then 2
    cplx vd[4];   // (dp, dm) for field value 1 then 2
    // the on-site field (src/dqmc_config_u), when lwrapu: conf_u [ltrot][n], values 1..ulcomp
    int lwrapu, lwrapv, ulcomp, uphase_from_conf;
    int32_t *uconf;
    cplx ub[4], ubi[4], ud[12], uratio[12];   // bmat, bmat_inv, delta_bmat(iflip, is), phase_ratio
    double ug[4], upa[4];                      // gaml, arg of phase(is)
    // the G-based updates of the on-site field: the slice's field before the update
    int32_t *uold;
};

// uniforms of one slice in a pass: 2 per site of the on-site field, 2 per bond of every family
__host__ __device__ __forceinline__ size_t p_slice_draws(const PChain &c)
{
    return (c.lwrapu ? (size_t)2 * c.n : 0) + (c.lwrapv ? (size_t)2 * c.nn_lf * c.nn_nf : 0);
}

__device__ __forceinline__ cplx *pmat(const PChain &c, int sel, int pt)
{
    const size_t nne = (size_t)c.n * c.ne;
    switch (sel) {
    case P_UR: return c.UR;
    case P_UL: return c.UL;
    case P_ULRINV: return c.ULRINV;
    case P_ULR: return c.ULR;
    case P_T1: return c.T1;
    case P_T2: return c.T2;
    case P_ULO: return c.ULo;
    case P_URO: return c.URo;
    case P_INV2: return c.INV2;
    case P_G: return c.G;
    case P_G2: return c.G2;
    case P_KT: return (cplx *)c.kt;
    case P_KTM1: return (cplx *)c.ktm1;
    case P_UST: return c.Ust + nne * pt;
    case P_PROJ: return c.proj;
    }
    return nullptr;
}

template <int NT, int NF>
__global__ void kp_stock_sites(const PChain *chains, int nt, int i0, int nup, size_t uoff);
template <int NT>
__global__ void kp_stock_bonds(const PChain *chains, int nt, int nf, int ib0, int nb, int uoff);
extern "C" __global__ void kp_stock_pre(const PChain *chains, int nch, int grp, int nf, int ib0, int nup);
extern "C" __global__ void kp_stock_f(const PChain *chains, int nch, int grp, int nf, int ib0, int nup);
extern "C" __global__ void kp_stock_vtmp(const PChain *chains, int nch, int grp, int nup);
extern "C" __global__ void kp_stock_flush(const PChain *chains, int nch, int grp, int nup);
