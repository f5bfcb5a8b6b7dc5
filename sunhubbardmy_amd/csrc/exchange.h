// exchange.h -- the sequential Metropolis decisions of a block of up to 64 sites of one chain, shared by
// every update that works on such a block: the on-site and bond fields of the finite-temperature sweep
// (blocks of G) and of the projective sweep (stocks of UR (UL UR)^-1 UL).
#pragma once
#include "sunhip_kernels.h"
#include <type_traits>

#define UB 64   // sites of a block

// a + b c
__device__ __forceinline__ cplx cfma(cplx a, cplx b, cplx c)
{
    return make_double2(fma(-b.y, c.y, fma(b.x, c.x, a.x)), fma(b.y, c.x, fma(b.x, c.y, a.y)));
}

// z times a power of two: the larger part in [1/2, 1)
__device__ __forceinline__ cplx pow2_unit(cplx z)
{
    const int k = -__builtin_amdgcn_frexp_exp(fmax(fabs(z.x), fabs(z.y)));
    return make_double2(ldexp(z.x, k), ldexp(z.y, k));
}

// The decisions of the block's sites 0 .. nb - 1, nb <= 16 NT, by a workgroup of NT waves.  Wave w holds the
// columns 16 w .. 16 w + 15 of the block H as NT accumulator tiles of the FP64 MFMA (element r of lane l:
// column l/16 + 4r, row l%16 of the tile).  Four sites g at a time, one barrier each: every wave
// reads the 4 x 4 block H_gg, decides the four sites (PAIR: the two bonds) one after the other, the same
// operations in every lane and no branches (a rejected site has sigma = 0), and H takes their
// product as one rank-4 MFMA update.  With sigma_k = delta / (1 + delta (1 - d_kk)) and the elimination
//   c_ik = sigma_k d_ik, d_ij += c_ik d_kj   (i, j > k)
// the product is H + H(:, g) x, x = T_g H(g, :) by the substitutions
//   b_k = r_k + sum_{l<k} c_kl b_l,  x_k = sigma_k (b_k + sum_{l>k} d_kl x_l).
// PAIR: sites 2q and 2q + 1 are one bond and flip together, ratio = det M with M = 1 + (1 - d_bb) diag(delta)
// and the 2 x 2 matrix diag(delta) M^-1 in place of sigma (its adjugate over the determinant, so that
// neither site needs a pivot of its own).
// WHOLE (the block is all of G, n <= 64): H is G, the rows are r = G(g, :) - E_g (each accepted site
// is G += sigma G(:, s) (G(s, :) - e_s)), and G is written back at the end.  Otherwise H starts as
// the block of G and takes exchange steps: the accepted rows and columns of H are cleared, the
// accepted rows of H(:, g) and columns of r replaced by unit vectors, so that
//   H_ij + H_iP T H_Pj,  H_iP T,  T H_Pj  and  T   (i, j outside P)
// stand in the four parts and H(P, P) ends as T = (diag(1/delta) + 1 - H(P, P))^-1 of the whole block.
// Bound by a serial chain per group, in cycles at NT = 4 (stamps in a copy): the four decisions 1300
// (about fifteen dependent FP64 operations and a hardware reciprocal each), the barrier and the LDS
// round trip 700, the substitutions 650, the wave's 16 MFMAs 1040, the publication 480.  One site at a
// time with the block spread over 16 x 16 threads takes 1360 cycles a site, 41 us a block against 30
// here: a barrier and eleven LDS reads per thread and site for one rank-1 update.
// Acceptance is |Re(ratiotot phase)| > u2 |Re(phase)| with ratiotot = ratio1^nflr qf: the
// reference's |Re(ratiotot phase) / Re(phase)| > u2 without the division.  Only the direction of phase
// counts; so that the accepted ratios of a block (1e200 for twelve flavours far from the weights' maximum) do not leave the
// exponent range, it takes an exact power of two after every group, and with nflr not known here (NF = 0)
// after every site (37.1 -> 38.0 us a block for 72 chains): neither decisions nor direction depend on it.
//
// P: load(i, j) the entry of the block; factors(site, db, qf, u2) of a site < nb, its delta, field-only
// factor and acceptance uniform (PAIR: qf and u2 of the bond's first site); store(i, j, v, ri, rj) for
// i, j < nb the final entry, ri, rj the places of i, j among the accepted sites or -1; finish(site, rank) for an
// accepted site, lane by lane of wave 0; done(ka, phase) by one thread.
template <int NT, bool WHOLE, bool PAIR, int NF, class P>
__device__ __forceinline__ void exchange_block(P &pol, int nb, int nflr, cplx phase)
{
    __shared__ cplx colb[2][4][UB], rowb[2][4][UB];
    __shared__ cplx sdb[UB + 4], sqf[UB + 4];
    __shared__ double su2[UB + 4];
    const int lane = threadIdx.x & 63, l16 = lane & 15, kq = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the same in every lane: scalar branches on it
    double4_t hr[NT], hi[NT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = 16 * t + l16, j = 16 * w + kq + 4 * r;
            const cplx g = pol.load(min(i, nb - 1), min(j, nb - 1));
            hr[t][r] = i < nb && j < nb ? g.x : 0.0;
            hi[t][r] = i < nb && j < nb ? g.y : 0.0;
        }
    // the factors that do not depend on H, site by site in LDS; past the block a site that is never accepted
    cplx fdb = make_double2(0.0, 0.0), fqf = make_double2(0.0, 0.0);
    double fu2 = __builtin_inf();
    if (w == 0 && lane < nb) pol.factors(lane, fdb, fqf, fu2);
    if (w == 0) {
        sdb[lane] = fdb;
        sqf[lane] = fqf;
        su2[lane] = fu2;
    }
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
        cplx g2[2][2][2];       // PAIR: diag(delta) M^-1 of each bond
        unsigned mg = 0;
        if constexpr (PAIR) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int k = 2 * q;
                const cplx dp = db[k], dm = db[k + 1];
                cplx m11 = cmul(make_double2(1.0 - d[k][k].x, -d[k][k].y), dp), m22 = cmul(make_double2(1.0 - d[k + 1][k + 1].x, -d[k + 1][k + 1].y), dm);
                m11.x += 1.0;
                m22.x += 1.0;
                const cplx m12 = cmul(make_double2(-d[k][k + 1].x, -d[k][k + 1].y), dm);
                const cplx m21 = cmul(make_double2(-d[k + 1][k].x, -d[k + 1][k].y), dp);
                const cplx ratio = csub(cmul(m11, m22), cmul(m12, m21));
                const cplx rt = cmul(ratio, cmul(phase, qf[k]));
                const double dd = cabs2(ratio);
                double rd = __builtin_amdgcn_rcp(dd);
                rd = fma(rd, fma(-dd, rd, 1.0), rd);
                rd = fma(rd, fma(-dd, rd, 1.0), rd);
                const cplx inv = cscale(cconj(ratio), rd), ip = cmul(dp, inv), im = cmul(dm, inv);
                cplx t[2][2] = {{cmul(m22, ip), cmul(make_double2(-m12.x, -m12.y), ip)},
                                {cmul(make_double2(-m21.x, -m21.y), im), cmul(m11, im)}};
                const bool acc = fabs(rt.x) > u2[k] * fabs(phase.x);
                phase.x = acc ? rt.x : phase.x;
                phase.y = acc ? rt.y : phase.y;
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        // (pinned: moved behind the decision, the two chains would run one after the other)
                        asm volatile("" : "+v"(t[i][j].x), "+v"(t[i][j].y));
                        g2[q][i][j].x = acc ? t[i][j].x : 0.0;
                        g2[q][i][j].y = acc ? t[i][j].y : 0.0;
                    }
                mg |= (__ballot(acc) != 0 ? 3u : 0u) << k;
                if (q == 0) {
                    // c = d(bond 1, bond 0) g, in place, and the second bond's block
#pragma unroll
                    for (int i = 2; i < 4; i++) {
                        const cplx c0 = cfma(cmul(d[i][0], g2[0][0][0]), d[i][1], g2[0][1][0]);
                        const cplx c1 = cfma(cmul(d[i][0], g2[0][0][1]), d[i][1], g2[0][1][1]);
                        d[i][0] = c0;
                        d[i][1] = c1;
#pragma unroll
                        for (int j = 2; j < 4; j++) d[i][j] = cfma(cfma(d[i][j], c0, d[0][j]), c1, d[1][j]);
                    }
                }
            }
        } else {
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
                if (NF == 0) phase = pow2_unit(phase);
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
        }
        if (PAIR || NF > 0) phase = pow2_unit(phase);
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
            if constexpr (PAIR) {
#pragma unroll
                for (int i = 2; i < 4; i++) rv[i] = cfma(cfma(rv[i], d[i][0], rv[0]), d[i][1], rv[1]);
                const cplx x2 = cfma(cmul(g2[1][0][0], rv[2]), g2[1][0][1], rv[3]), x3 = cfma(cmul(g2[1][1][0], rv[2]), g2[1][1][1], rv[3]);
                const cplx y0 = cfma(cfma(rv[0], d[0][2], x2), d[0][3], x3), y1 = cfma(cfma(rv[1], d[1][2], x2), d[1][3], x3);
                rv[0] = cfma(cmul(g2[0][0][0], y0), g2[0][0][1], y1);
                rv[1] = cfma(cmul(g2[0][1][0], y0), g2[0][1][1], y1);
                rv[2] = x2;
                rv[3] = x3;
            } else {
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
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = 16 * t + l16, j = 16 * w + kq + 4 * r;
            if (i < nb && j < nb)
                pol.store(i, j, make_double2(hr[t][r], hi[t][r]), mask >> i & 1 ? rank(i) : -1, mask >> j & 1 ? rank(j) : -1);
        }
    if (w == 0 && lane < nb && (mask >> lane & 1)) pol.finish(lane, rank(lane));
    if (threadIdx.x == 0) pol.done(ka, cscale(phase, 1.0 / sqrt(cabs2(phase))));
}
