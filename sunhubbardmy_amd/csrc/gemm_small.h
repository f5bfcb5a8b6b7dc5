// gemm_small.h -- complex product on one 32 x 32 tile (FP64 MFMA), for launches that would leave most of the
// chip without a 64 x 64 tile.  Each of the workgroup's four waves holds the whole tile and takes every
// fourth step of K, operands straight from L2 in the MFMA layout, four steps' loads ahead of the
// MFMAs; the waves' sums meet in LDS, where wave w adds up and stores the w-th 16 x 16 part.
// Bound by the wave's MFMAs (64 cycles each, 16 per step of 4) and one round trip to L2 per 64 of K.  One product
// of N = 288: 56 us on 25 64 x 64 tiles, 18 on 81 of these; 64 x 324 x 324 for eight chains 57 -> 16 us.
#pragma once
#include "sunhip_kernels.h"

#define GS 32

// Products deal a batch's tiles out in groups of grp chains, tile after tile, so that with eight a chain's
// tiles share one XCD (workgroups go round the eight XCDs in launch order) and its L2 holds the operands once
// instead of every L2 a part of each.  tiles: of the largest chain
__device__ __forceinline__ bool tile_of(int tiles, int nch, int grp, int &chain, int &tile)
{
    const int g = blockIdx.x / (grp * tiles), q = blockIdx.x % (grp * tiles);
    chain = g * grp + q % grp;
    tile = q / grp;
    return chain < nch;
}
// (a batch that is no multiple of eight has idle places in its last group: few chains go as one group)
__host__ inline int tile_group(int nch) { return nch % 8 == 0 || nch > 32 ? 8 : nch; }
__host__ inline unsigned tile_grid(int tiles, int nch) { return (unsigned)((nch - 1) / tile_group(nch) + 1) * tile_group(nch) * tiles; }

// la(row, k), lb(k, col): entries of the operands, row and col within the tile of 16 HM x 16 HN (past the edge any
// valid entry); k < kk is checked here.  st(row, col, v) gets every entry of the tile.
template <int HM, int HN, class LA, class LB, class ST>
__device__ __forceinline__ void gemm_small_tile(int kk, LA la, LB lb, ST st)
{
    constexpr int P = HM * HN;      // wave w sums up and stores the slices w P .. of the 4 P (part, element) slices
    __shared__ cplx red[4 * P][3][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, lq = lane >> 4;
    double4_t accr[HM][HN] = {}, acci[HM][HN] = {};     // transposed 16 x 16 tiles
    cplx ya[4][HM], xa[4][HN];
    auto load = [&](int k0) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int k = k0 + 16 * s + 4 * w + lq, kc = min(k, kk - 1);
            const bool in = k < kk;
#pragma unroll
            for (int h = 0; h < HM; h++) {
                const cplx a = la(16 * h + l16, kc);
                ya[s][h] = make_double2(in ? a.x : 0.0, in ? a.y : 0.0);
            }
#pragma unroll
            for (int h = 0; h < HN; h++) {
                const cplx b = lb(kc, 16 * h + l16);
                xa[s][h] = make_double2(in ? b.x : 0.0, in ? b.y : 0.0);
            }
        }
    };
    load(0);
    for (int k0 = 0; k0 < kk; k0 += 64) {
        cplx y[4][HM], x[4][HN];
#pragma unroll
        for (int s = 0; s < 4; s++) {
#pragma unroll
            for (int h = 0; h < HM; h++) y[s][h] = ya[s][h];
#pragma unroll
            for (int h = 0; h < HN; h++) x[s][h] = xa[s][h];
        }
        if (k0 + 64 < kk) load(k0 + 64);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (k0 + 16 * s + 4 * w >= kk) break;
#pragma unroll
            for (int sm = 0; sm < HM; sm++)
#pragma unroll
                for (int sn = 0; sn < HN; sn++) {
                    accr[sm][sn] = mfma(x[s][sn].x, y[s][sm].x, accr[sm][sn]);
                    acci[sm][sn] = mfma(x[s][sn].x, y[s][sm].y, acci[sm][sn]);
                    accr[sm][sn] = mfma(-x[s][sn].y, y[s][sm].y, accr[sm][sn]);
                    acci[sm][sn] = mfma(x[s][sn].y, y[s][sm].x, acci[sm][sn]);
                }
        }
    }
    // slice 4 o + r: element r of part o = sm + HM sn
#pragma unroll
    for (int q = 0; q < 4 * P; q++)
        if (q / P != w)
            red[q][w < q / P ? w : w - 1][lane] = make_double2(accr[(q >> 2) % HM][(q >> 2) / HM][q & 3], acci[(q >> 2) % HM][(q >> 2) / HM][q & 3]);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4 * P; q++)
        if (q / P == w) {
            cplx v = make_double2(accr[(q >> 2) % HM][(q >> 2) / HM][q & 3], acci[(q >> 2) % HM][(q >> 2) / HM][q & 3]);
#pragma unroll
            for (int p = 0; p < 3; p++) v = cadd(v, red[q][p][lane]);
            st(16 * ((q >> 2) % HM) + l16, 16 * ((q >> 2) / HM) + lq + 4 * (q & 3), v);
        }
}

// one 32 x 32 tile (tm, tn) of C (m x n, ldc) = alpha op(A) op(B) + beta C; op = 0: as stored, 1: conjugate
// transpose
template <int OPA, int OPB>
__device__ __forceinline__ void zgemm_small(const cplx *A_, int lda, const cplx *B_, int ldb, cplx *C_, int ldc, int m, int n,
                                            int kk, int tm, int tn, double ar, double ai, double br, double bi)
{
    GAS cplx *A = gp(A_), *B = gp(B_), *C = gp(C_);
    const bool zb = (br == 0.0 && bi == 0.0);
    gemm_small_tile<2, 2>(
        kk,
        [=](int i, int k) {
            const int row = min(tm + i, m - 1);
            return OPA == 0 ? gld(A + ((size_t)row + (size_t)k * lda)) : cconj(gld(A + ((size_t)k + (size_t)row * lda)));
        },
        [=](int k, int j) {
            const int col = min(tn + j, n - 1);
            return OPB == 0 ? gld(B + ((size_t)k + (size_t)col * ldb)) : cconj(gld(B + ((size_t)col + (size_t)k * ldb)));
        },
        [=](int i, int j, cplx v) {
            const int row = tm + i, col = tn + j;
            if (row >= m || col >= n) return;
            const size_t e = (size_t)row + (size_t)col * ldc;
            double outr = ar * v.x - ai * v.y, outi = ar * v.y + ai * v.x;
            if (!zb) { const cplx cv = gld(C + e); outr += br * cv.x - bi * cv.y; outi += br * cv.y + bi * cv.x; }
            gst(C + e, make_double2(outr, outi));
        });
}

