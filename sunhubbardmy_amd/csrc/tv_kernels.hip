// tv_kernels.hip -- the bond field of the finite-temperature t-V model (vconf, lprojv = .false.):
// the per-bond 2x2 props of one family on rows or columns of a chain matrix
// (src/dqmc_config_v/dqmc_{left,right}_{forward,backward}_prop.f90).  The field of bond q of
// family nf at slice nt is confv[((nt - 1) nn_nf + nf) n + q] (1 or 2); u = ut = [[1, 1],
// [1, -1]] / sqrt(2); vtb = (bp, bm, bpi, bmi) of component 1 then 2, vdl = (dp, dm) of 1 then 2.
#pragma once

#define V_S 0.70710678118654752440

// rows (side 0) or columns (side 1) i1, i2 of every bond of family nf, one (bond, index) per
// thread:
//   rows: mode 0 diag(bp, bm) ut (left_forward nflag 2), 1 u (left_forward nflag 1,
//         left_backward nflag 2), 2 u diag(bpi, bmi) (left_backward nflag 1)
//   cols: mode 0 (. u) diag(bpi, bmi) (right_backward nflag 2), 1 . u (right_backward nflag 1,
//         right_forward nflag 2), 2 (. diag(bp, bm)) ut (right_forward nflag 1)
extern "C" __global__ void __launch_bounds__(256)
k_vprop(const DChain *chains, int msel, int pt, int nf, int mode, int side, int nt)
{
    const DChain &c = chains[blockIdx.z];
    if (!c.lwrapv) return;
    const int n = c.n, nl = c.nn_lf;
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= n * nl) return;
    const int q = side ? e / n : e % nl, j = side ? e % n : e / nl;
    const int ist = nf * nl + q;
    const int i1 = c.bonds[2 * ist], i2 = c.bonds[2 * ist + 1];
    const int is = c.confv[((size_t)(nt - 1) * c.nn_nf + nf) * n + q] - 1;
    GAS cplx *M = gp(chain_mat(c, msel, pt));
    GAS cplx *px = side ? M + (size_t)i1 * n + j : M + (size_t)j * n + i1;
    GAS cplx *py = side ? M + (size_t)i2 * n + j : M + (size_t)j * n + i2;
    cplx x = gld(px), y = gld(py);
    const cplx bp = c.vtb[4 * is], bm = c.vtb[4 * is + 1], bpi = c.vtb[4 * is + 2], bmi = c.vtb[4 * is + 3];
    if (mode == 2) {
        x = cmul(side ? bp : bpi, x);
        y = cmul(side ? bm : bmi, y);
    }
    cplx v1 = cscale(cadd(x, y), V_S), v2 = cscale(csub(x, y), V_S);
    if (mode == 0) {
        v1 = cmul(side ? bpi : bp, v1);
        v2 = cmul(side ? bmi : bm, v2);
    }
    gst(px, v1);
    gst(py, v2);
}

