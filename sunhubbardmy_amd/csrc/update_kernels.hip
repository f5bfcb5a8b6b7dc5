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
// chip.  Per slice: one N = 288 chain 1.72 -> 0.27 ms, 72 chains of N = 64, 144, 256 0.90 -> 0.29 ms,
// 256 chains of N = 256 1.20 -> 0.95 ms (per block 40 us of decisions, 55 us of panels, 140 us of
// flush; one read and write of the 256 MiB of G takes 111 us), 16 chains of N = 64 172 -> 31 us.
#include "update_kernels.h"
#include <type_traits>

// lane l's value as a wave-uniform one; l must be wave-uniform
__device__ __forceinline__ double lane_d(double v, int l)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l), __builtin_amdgcn_readlane(__double2loint(v), l));
}
__device__ __forceinline__ cplx lane_c(cplx v, int l) { return make_double2(lane_d(v.x, l), lane_d(v.y, l)); }
// a + b c
__device__ __forceinline__ cplx cfma(cplx a, cplx b, cplx c)
{
    return make_double2(fma(-b.y, c.y, fma(b.x, c.x, a.x)), fma(b.y, c.x, fma(b.x, c.y, a.y)));
}

// The decisions of sites s0 .. s0 + nb - 1, nb <= 16 NT.  Wave w of the NT waves holds the columns
// 16 w .. 16 w + 15 of the block H as NT accumulator tiles of the FP64 MFMA (element r of lane l:
// column l/16 + 4r, row l%16 of the tile).  Four sites g at a time, one barrier each: every wave
// reads the 4 x 4 block H_gg, decides the four sites one after the other (the same operations in
// every lane, no branches: a rejected site has sigma = 0), and H takes the four sites' product as
// one rank-4 MFMA update.  With sigma_k = delta / (1 + delta (1 - d_kk)) and the elimination
//   c_ik = sigma_k d_ik, d_ij += c_ik d_kj   (i, j > k)
// the product is H + H(:, g) x, x = T_g H(g, :) by the substitutions
//   b_k = r_k + sum_{l<k} c_kl b_l,  x_k = sigma_k (b_k + sum_{l>k} d_kl x_l).
// WHOLE (the block is all of G, n <= 64): H is G, the rows are r = G(g, :) - E_g (each accepted site
// is G += sigma G(:, s) (G(s, :) - e_s)), and G is written back at the end.  Otherwise H starts as
// the block of G and takes exchange steps: the accepted rows and columns of H are cleared, the
// accepted rows of H(:, g) and columns of r replaced by unit vectors, so that
//   H_ij + H_iP T H_Pj,  H_iP T,  T H_Pj  and  T   (i, j outside P)
// stand in the four parts and H(P, P) ends as T of the whole block.
// Bound by a serial chain per group, in cycles at NT = 4 (stamps in a copy): the four decisions 1300
// (about fifteen dependent FP64 operations and a hardware reciprocal each), the barrier and the LDS
// round trip 700, the substitutions 650, the wave's 16 MFMAs 1040, the publication 480.  One site at a
// time with the block spread over 16 x 16 threads takes 1360 cycles a site, 41 us a block against 30
// here: a barrier and eleven LDS reads per thread and site for one rank-1 update.
// Acceptance is |Re(ratiotot phase)| > u2 |Re(phase)| with ratiotot = ratio1^nflr qf: the
// reference's |Re(ratiotot phase) / Re(phase)| > u2 without the division, which lets phase grow
// unnormalised over the block.
template <int NT, bool WHOLE, int NF>
__global__ void __launch_bounds__(64 * NT, 2)
k_upd_sites(const DChain *chains, int nt, int slice_in_pass, int s0)
{
    __shared__ cplx colb[2][4][UB], rowb[2][4][UB];
    __shared__ cplx sdb[UB + 4], sqf[UB + 4];
    __shared__ double su2[UB + 4];
    const DChain &c = chains[blockIdx.x];
    const int n = c.n;
    if (s0 >= n) return;
    const int nb = min(16 * NT, n - s0);
    const int lane = threadIdx.x & 63, l16 = lane & 15, kq = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the same in every lane: scalar branches on it
    GAS cplx *G = gp(c.G) + ((size_t)s0 + (size_t)s0 * n);
    double4_t hr[NT], hi[NT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = 16 * t + l16, j = 16 * w + kq + 4 * r;
            const cplx g = gld(G + ((size_t)min(i, nb - 1) + (size_t)min(j, nb - 1) * n));
            hr[t][r] = i < nb && j < nb ? g.x : 0.0;
            hi[t][r] = i < nb && j < nb ? g.y : 0.0;
        }
    // lane l of every wave holds the factors of site l that do not depend on G: delta, gaml(isp) /
    // gaml(is) phase_ratio and the acceptance uniform; past the block a site that is never accepted
    int32_t *cf = c.conf + (size_t)(nt - 1) * n + s0;
    cplx fdb = make_double2(0.0, 0.0), fqf = make_double2(0.0, 0.0);
    double fu2 = __builtin_inf();
    int fisp = 1;
    if (lane < nb) {
        const double *u = c.unif + (size_t)2 * n * slice_in_pass + 2 * (s0 + lane);
        const int is = cf[lane], fl = (int)ceil(u[0] * (c.lcomp - 1));
        fisp = (is + fl - 1) % c.lcomp + 1;
        const int k = (fl - 1) + (c.lcomp - 1) * (is - 1);
        fdb = c.delta_bmat[k];
        fqf = cscale(c.phase_ratio[k], c.gaml[fisp - 1] / c.gaml[is - 1]);
        fu2 = u[1];
    }
    if (w == 0) {
        sdb[lane] = fdb;
        sqf[lane] = fqf;
        su2[lane] = fu2;
    }
    const int nflr = c.nflr;
    cplx db[4], qf[4];
    double u2[4];
    auto factors = [&](int s) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            db[k] = sdb[s + k];
            qf[k] = sqf[s + k];
            u2[k] = su2[s + k];
        }
    };
    cplx phase = make_double2(c.sc[SC_PHASE], c.sc[SC_PHASE + 1]);
    unsigned long long mask = 0;
    // columns 16 T + 4 X .. + 3 (held by wave T) and the same rows (tile T of every wave)
    auto publish = [&](int T, auto X, int buf) {
        constexpr int x = decltype(X)::value;
        if (w == T)
#pragma unroll
            for (int t = 0; t < NT; t++) colb[buf][kq][16 * t + l16] = make_double2(hr[t][x], hi[t][x]);
#pragma unroll
        for (int t = 0; t < NT; t++)
            if (t == T && (l16 >> 2) == x)
#pragma unroll
                for (int r = 0; r < 4; r++) rowb[buf][l16 & 3][16 * w + kq + 4 * r] = make_double2(hr[t][r], hi[t][r]);
    };
    auto group = [&](int T, auto X) {
        constexpr int x = decltype(X)::value;
        const int s = 16 * T + 4 * x, buf = x & 1;
        __syncthreads();
        cplx d[4][4], rv[4], cv[NT];
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) d[i][j] = colb[buf][j][s + i];
#pragma unroll
        for (int k = 0; k < 4; k++) rv[k] = rowb[buf][k][16 * w + l16];
#pragma unroll
        for (int t = 0; t < NT; t++) cv[t] = colb[buf][kq][16 * t + l16];
        cplx sg[4];
        unsigned mg = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            // ratio1 = 1 + delta - delta G(s, s)
            const cplx g = d[k][k], dk = db[k];
            const cplx r1 = make_double2(fma(dk.y, g.y, fma(-dk.x, g.x, 1.0 + dk.x)), fma(-dk.y, g.x, fma(-dk.x, g.y, dk.y)));
            cplx rt = cmul(r1, cmul(phase, qf[k]));
            if (NF > 0) {
#pragma unroll
                for (int f = 1; f < NF; f++) rt = cmul(rt, r1);
            } else {
                for (int f = 1; f < nflr; f++) rt = cmul(rt, r1);
            }
            // sigma = delta conj(ratio1) / |ratio1|^2, the reciprocal by two Newton steps on the
            // hardware's estimate (|ratio1|^2 is far from the ends of the exponent range)
            const double dd = cabs2(r1);
            double rd = __builtin_amdgcn_rcp(dd);
            const double re = fma(-dd, rd, 1.0);
            rd = fma(rd, fma(re, re, re), rd);
            cplx sk = cscale(cmul(dk, cconj(r1)), rd);
            // (pinned here: moved behind the decision, the two chains would run one after the other)
            asm volatile("" : "+v"(sk.x), "+v"(sk.y));
            const bool acc = fabs(rt.x) > u2[k] * fabs(phase.x);
            phase.x = acc ? rt.x : phase.x;
            phase.y = acc ? rt.y : phase.y;
            sg[k].x = acc ? sk.x : 0.0;
            sg[k].y = acc ? sk.y : 0.0;
            mg |= (__ballot(acc) != 0 ? 1u : 0u) << k;
#pragma unroll
            for (int i = k + 1; i < 4; i++) {
                d[i][k] = cmul(sg[k], d[i][k]);
#pragma unroll
                for (int j = k + 1; j < 4; j++) d[i][j] = cfma(d[i][j], d[i][k], d[k][j]);
            }
        }
        factors(min(s + 4, UB - 4));   // the next group's, on their way while this one is applied
        if (mg != 0) {
            mask |= (unsigned long long)mg << s;
            // lane l16's place in the group, as a row of tile T or a column of wave T
            const int q = l16 - 4 * x;
            const bool in = (unsigned)q < 4u, ain = in && (mg >> q & 1);
            if (WHOLE) {
                if (w == T)
#pragma unroll
                    for (int k = 0; k < 4; k++) rv[k].x -= q == k ? 1.0 : 0.0;
            } else {
                if (w == T) {
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        rv[k].x = ain ? (q == k ? 1.0 : 0.0) : rv[k].x;
                        rv[k].y = ain ? 0.0 : rv[k].y;
                    }
                    const bool ac = mg >> kq & 1;
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        hr[t][x] = ac ? 0.0 : hr[t][x];
                        hi[t][x] = ac ? 0.0 : hi[t][x];
                    }
                }
#pragma unroll
                for (int t = 0; t < NT; t++)
                    if (t == T) {
                        cv[t].x = ain ? (q == kq ? 1.0 : 0.0) : cv[t].x;
                        cv[t].y = ain ? 0.0 : cv[t].y;
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            hr[t][r] = ain ? 0.0 : hr[t][r];
                            hi[t][r] = ain ? 0.0 : hi[t][r];
                        }
                    }
            }
#pragma unroll
            for (int k = 1; k < 4; k++)
#pragma unroll
                for (int l = 0; l < k; l++) rv[k] = cfma(rv[k], d[k][l], rv[l]);
#pragma unroll
            for (int k = 3; k >= 0; k--) {
#pragma unroll
                for (int l = k + 1; l < 4; l++) rv[k] = cfma(rv[k], d[k][l], rv[l]);
                rv[k] = cmul(sg[k], rv[k]);
            }
            const cplx xa = kq & 1 ? rv[1] : rv[0], xb = kq & 1 ? rv[3] : rv[2], xv = kq & 2 ? xb : xa;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                hr[t] = mfma(xv.x, cv[t].x, hr[t]);
                hi[t] = mfma(xv.x, cv[t].y, hi[t]);
            }
#pragma unroll
            for (int t = 0; t < NT; t++) {
                hr[t] = mfma(-xv.y, cv[t].y, hr[t]);
                hi[t] = mfma(xv.y, cv[t].x, hi[t]);
            }
        }
        if constexpr (x < 3)
            publish(T, std::integral_constant<int, x + 1>(), buf ^ 1);
        else if (T + 1 < NT)
            publish(T + 1, std::integral_constant<int, 0>(), buf ^ 1);
    };
    publish(0, std::integral_constant<int, 0>(), 0);
    __syncthreads();
    factors(0);
#pragma unroll
    for (int T = 0; T < NT; T++) {
        if (16 * T >= nb) break;
        group(T, std::integral_constant<int, 0>());
        group(T, std::integral_constant<int, 1>());
        group(T, std::integral_constant<int, 2>());
        group(T, std::integral_constant<int, 3>());
    }
    const int ka = __popcll(mask);
    auto rank = [&](int i) { return __popcll(mask & ((1ull << i) - 1)); };
    GAS cplx *T = WHOLE ? G : gp(c.updt);
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = 16 * t + l16, j = 16 * w + kq + 4 * r;
            const cplx v = make_double2(hr[t][r], hi[t][r]);
            if (WHOLE) {
                if (i < nb && j < nb) gst(T + ((size_t)i + (size_t)j * n), v);
            } else if ((mask >> i & 1) && (mask >> j & 1)) {
                gst(T + (rank(i) + UB * rank(j)), v);
            }
        }
    if (w == 0 && lane < nb && (mask >> lane & 1)) {
        cf[lane] = fisp;
        if (!WHOLE) c.updp[1 + rank(lane)] = s0 + lane;
    }
    if (threadIdx.x == 0) {
        if (!WHOLE) c.updp[0] = ka;
        phase = cscale(phase, 1.0 / sqrt(cabs2(phase)));
        c.sc[SC_PHASE] = phase.x;
        c.sc[SC_PHASE + 1] = phase.y;
        c.sc[SC_ACC] += ka;
        c.sc[SC_TRIED] += nb;
    }
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

#endif

// one object file per (WHOLE, NF) pair, so that they compile side by side
template __global__ void k_upd_sites<1, UPD_WHOLE, UPD_NF>(const DChain *, int, int, int);
template __global__ void k_upd_sites<2, UPD_WHOLE, UPD_NF>(const DChain *, int, int, int);
template __global__ void k_upd_sites<3, UPD_WHOLE, UPD_NF>(const DChain *, int, int, int);
template __global__ void k_upd_sites<4, UPD_WHOLE, UPD_NF>(const DChain *, int, int, int);
