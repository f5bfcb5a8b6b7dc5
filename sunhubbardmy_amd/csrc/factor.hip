// factor.hip -- QR, Q formation and LU of the chains' N x N matrices, N <= 512, spread over the chip:
// a workgroup of NW waves owns 16 columns of one chain's matrix, all rows, in registers.
//
// Layout: wave w holds the 16-row tiles w, w + NW, ... of its 16 columns as FP64 MFMA accumulators
// (lane l, element r of a tile: row 4 r + l/16, column l%16).  The same registers serve as B operand
// of V^H X (K index = row) and, for a block that is a panel itself, hold everything a column-by-column
// factorization touches, so a panel never leaves its registers.
//
//   k_qr_step(k)   Householder QR (zgeqrf + zlarft) one panel at a time: the workgroups of the column
//                  blocks >= k apply panel k - 1, and the one that owns block k goes on to factor it.
//                  The trailing blocks and the next panel share a launch, one launch per panel.
//   k_formq_cb     Q = H_1 ... H_n (zungqr): the columns of Q are independent, so every workgroup takes
//                  its 16 columns of the identity through the panels, in one launch.
//   k_lu_step(k)   LU with partial pivoting (zgetrf), panels and trailing blocks as in k_qr_step; the
//                  interchanges of panel k - 1 reach the blocks right of it as a permuted load, the
//                  blocks left of it in one last launch.
//
// The grid is chains x blocks, so that the panels, the longest workgroups, start first, and a batch of a
// multiple of eight chains keeps a chain's blocks on one XCD, whose L2 then holds the panel they share.
//
// Bound by the chain of panels: about 1.3 us a column (in a QR panel of 64 rows, cycles per column: broadcast
// and dot products 800, sums over the wave and behind the barrier 700, the scalars 500, the update 450)
// and 5 us a launch for the operands' round trips and the rank-16 product; for 256 chains the trailing
// blocks' reads and writes. One workgroup per chain with LDS panels took 8 us a column. Measured, QR / LU of a
// batch: 16 chains of N = 64 296 -> 105 / 194 -> 150 us, 8 of N = 144 806 -> 242 / 508 -> 342, one of N = 288
// 2360 -> 659 / 1460 -> 960, 16 of N = 400 4500 -> 1010 / 2750 -> 1400, 256 of N = 256 2080 -> 1300 /
// 1550 -> 1340; Q: 256 of N = 256 1240 -> 680, one of N = 288 1220 -> 104. Broadcasting a column through LDS
// instead of the row lanes costs 1300 cycles a column more.
// Tall matrices (N x nc, the projective sweep's propagators, N <= 1024): the same kernels with nc columns; above 512 rows
// a wave holds eight tiles and broadcasts a column twice instead of keeping it.  Eight of 648 x 324: QR 1.6 ms and
// Q 0.25 (14.8 together in one workgroup per chain), the inverse of 324 x 324 1.3 ms (4.5).
#include "factor.h"
#include <type_traits>

// 1 / z: conj(z) / |z|^2 on z scaled by a power of two, the reciprocal by two Newton steps on the hardware's
// estimate (the compiled division takes about ten dependent operations, Smith's form three of them)
__device__ __forceinline__ cplx cinv_s(cplx z)
{
    const int k = -__builtin_amdgcn_frexp_exp(fmax(fabs(z.x), fabs(z.y)));
    const double x = ldexp(z.x, k), y = ldexp(z.y, k), d = fma(x, x, y * y);
    double r = __builtin_amdgcn_rcp(d);
    r = fma(r, fma(-d, r, 1.0), r);
    r = fma(r, fma(-d, r, 1.0), r);
    return make_double2(ldexp(x * r, k), ldexp(-y * r, k));
}

// lane J of every row group (16 lanes) to the whole group
template <int J>
__device__ __forceinline__ double row_bcast(double v)
{
    return dpp_d<0x150 + J>(v);     // row_newbcast:J
}

// f(0), f(1), ..., f(15) with compile-time arguments
template <int J = 0, class F>
__device__ __forceinline__ void cols16(F f)
{
    if constexpr (J < FPB) {
        f(std::integral_constant<int, J>());
        cols16<J + 1>(f);
    }
}

template <int FT>
struct FBlk {
    double4_t r[FT], i[FT];
};

// rows row0 + 16 rt + 4 r + l/16 (rt = w + NW tt) of column col0 + l%16; zero past nrow and ncol
template <int NW, int FT>
__device__ __forceinline__ void blk_load(FBlk<FT> &x, GAS cplx *A, int lda, int nrow, int col, int ncol, int w, int lq,
                                         const GAS int32_t *pm)
{
    const size_t cc = (size_t)min(col, ncol - 1) * lda;
#pragma unroll
    for (int tt = 0; tt < FT; tt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = 16 * (w + NW * tt) + 4 * r + lq, rc = min(row, nrow - 1);
            const cplx v = gld(A + ((size_t)(pm ? pm[rc] : rc) + cc));
            x.r[tt][r] = row < nrow && col < ncol ? v.x : 0.0;
            x.i[tt][r] = row < nrow && col < ncol ? v.y : 0.0;
        }
}

// entry (row, p) of a Householder panel stored LAPACK-style (unit diagonal implicit, zeros above)
__device__ __forceinline__ cplx panel_v(GAS cplx *V, int lda, int m, int b, int row, int p)
{
    const cplx v = gld(V + ((size_t)min(row, m - 1) + (size_t)min(p, b - 1) * lda));
    const bool in = row < m && p < b;
    return make_double2(in && row > p ? v.x : in && row == p ? 1.0 : 0.0, in && row > p ? v.y : 0.0);
}

// X <- (I - V op(T) V^H) X with the panel V (m x b, first row at tile toff of the workgroup's rows);
// op = conjugate transpose for HERM.  red: NW x 256 complex.  One barrier; red is free for the next
// use after the caller's next barrier (callers alternate between two).
template <int NW, bool HERM, int FT>
__device__ __forceinline__ void apply_panel(FBlk<FT> &x, GAS cplx *V, int lda, int m, int b, const GAS cplx *T, int toff, cplx *red,
                                            int w, int lane, int lq, int l16)
{
    double4_t wr = {}, wi = {};
#pragma unroll
    for (int tt = 0; tt < FT; tt++) {
        const int rt = w + NW * tt - toff;
        if (rt >= 0 && 16 * rt < m) {
            cplx v[4];
#pragma unroll
            for (int s = 0; s < 4; s++) v[s] = panel_v(V, lda, m, b, 16 * rt + 4 * s + lq, l16);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                wr = mfma(v[s].x, x.r[tt][s], wr);
                wi = mfma(v[s].x, x.i[tt][s], wi);
                wr = mfma(v[s].y, x.i[tt][s], wr);
                wi = mfma(-v[s].y, x.r[tt][s], wi);
            }
        }
    }
    cplx tv[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int kk = 4 * s + lq;
        const cplx t = gld(T + (HERM ? l16 * FPB + kk : kk * FPB + l16));   // conj T[kk][l16] or T[l16][kk]
        tv[s] = make_double2(t.x, HERM ? -t.y : t.y);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) red[w * 256 + r * 64 + lane] = make_double2(wr[r], wi[r]);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; r++) {
        cplx s = red[r * 64 + lane];
#pragma unroll
        for (int q = 1; q < NW; q++) s = cadd(s, red[q * 256 + r * 64 + lane]);
        wr[r] = s.x;
        wi[r] = s.y;
    }
    double4_t yr = {}, yi = {};
#pragma unroll
    for (int s = 0; s < 4; s++) {
        yr = mfma(tv[s].x, wr[s], yr);
        yi = mfma(tv[s].x, wi[s], yi);
        yr = mfma(-tv[s].y, wi[s], yr);
        yi = mfma(tv[s].y, wr[s], yi);
    }
#pragma unroll
    for (int tt = 0; tt < FT; tt++) {
        const int rt = w + NW * tt - toff;
        if (rt >= 0 && 16 * rt < m) {
            cplx v[4];
#pragma unroll
            for (int s = 0; s < 4; s++) v[s] = panel_v(V, lda, m, b, 16 * rt + l16, 4 * s + lq);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                x.r[tt] = mfma(-v[s].x, yr[s], x.r[tt]);
                x.i[tt] = mfma(-v[s].x, yi[s], x.i[tt]);
                x.r[tt] = mfma(v[s].y, yi[s], x.r[tt]);
                x.i[tt] = mfma(-v[s].y, yr[s], x.i[tt]);
            }
        }
    }
}

__device__ __forceinline__ cplx sum_lq(cplx v)
{
    v.x += swap16_d(v.x);
    v.y += swap16_d(v.y);
    v.x += swap32_d(v.x);
    v.y += swap32_d(v.y);
    return v;
}

template <int NW>
struct QrLds {
    cplx part[2][NW][16], rowj[2][16], S[FPB * FPB];
};

// Householder QR of the panel in x (b columns; its row 0 is row 0 of tile toff): column by column, the
// dot products of column j with every column come from one reduction (column j broadcast along the
// row groups of a wave through LDS, sums over the wave by lane swaps, over the waves through LDS
// behind the only barrier).  Columns q > j give v_j^H a_q for the update, columns q < j v_j^H v_q for
// T.  Every lane evaluates the scalars of zlarfg.  A column stays unscaled until the end (its lanes
// keep the factor), with alpha - beta in place of its row j while it is applied, so that the loop
// has no per-element cases outside the panel's first tile.
template <int NW, int FT>
__device__ __forceinline__ void qr_panel(FBlk<FT> &x, int b, int toff, cplx &tau_own, QrLds<NW> &L, int w, int lane, int lq, int l16)
{
    // of the lane's own column l16
    tau_own = make_double2(0.0, 0.0);
    cplx scal_own = make_double2(1.0, 0.0);
    double beta_own = 0.0;
    cols16([&](auto jc) {
        constexpr int j = decltype(jc)::value, par = j & 1;
        if (j >= b) return;
        if (w == toff && lq == (j & 3)) L.rowj[par][l16] = make_double2(x.r[0][j >> 2], x.i[0][j >> 2]);
        // column j along the row groups; of tile tt = 0 only the rows below row j (the other tiles of the
        // wave always lie below)
        cplx vb[FT > FTW ? 1 : FT][4], s0 = make_double2(0.0, 0.0), s1 = s0;
#pragma unroll
        for (int tt = 0; tt < FT; tt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                cplx v = make_double2(row_bcast<j>(x.r[tt][r]), row_bcast<j>(x.i[tt][r]));
                if (tt == 0) {
                    const bool in = w > toff || (w == toff && 4 * r + lq > j);
                    v.x = in ? v.x : 0.0;
                    v.y = in ? v.y : 0.0;
                }
                if (FT <= FTW || tt == 0) vb[tt][r] = v;
                cplx &s = r & 1 ? s1 : s0;
                s.x = fma(v.x, x.r[tt][r], fma(v.y, x.i[tt][r], s.x));
                s.y = fma(v.x, x.i[tt][r], fma(-v.y, x.r[tt][r], s.y));
            }
        cplx s = sum_lq(cadd(s0, s1));
        if (lq == 0) L.part[par][w][l16] = s;
        __syncthreads();
        s = L.part[par][0][l16];
#pragma unroll
        for (int q = 1; q < NW; q++) s = cadd(s, L.part[par][q][l16]);
        const double s2 = row_bcast<j>(s.x);
        const cplx ajq = L.rowj[par][l16], alpha = make_double2(row_bcast<j>(ajq.x), row_bcast<j>(ajq.y));
        cplx tau = make_double2(0.0, 0.0), scal = make_double2(1.0, 0.0), amb = make_double2(1.0, 0.0);
        double beta = alpha.x;
        if (!(s2 == 0.0 && alpha.y == 0.0)) {
            // the norm and its reciprocal from one Newton iteration for 1 / sqrt
            const double n2 = alpha.x * alpha.x + alpha.y * alpha.y + s2;
            double rs = __builtin_amdgcn_rsq(n2);
            rs = fma(rs, 0.5 * fma(-n2 * rs, rs, 1.0), rs);
            rs = fma(rs, 0.5 * fma(-n2 * rs, rs, 1.0), rs);
            double nrm = n2 * rs;
            nrm = fma(0.5 * rs, fma(-nrm, nrm, n2), nrm);
            beta = alpha.x >= 0 ? -nrm : nrm;
            const double ib = alpha.x >= 0 ? -rs : rs;
            amb = make_double2(alpha.x - beta, alpha.y);
            tau = make_double2(-amb.x * ib, -amb.y * ib);
            scal = cinv_s(amb);     // scaled: |alpha - beta|^2 leaves the exponent range before n2 does
        }
        // v_j^H (column l16): the sum over the rows below j in units of the unscaled column j
        const cplx wq = cadd(cmul(cconj(scal), s), ajq);
        if (w == 0 && lq == 0 && l16 < j) L.S[j * FPB + l16] = cconj(cmul(scal_own, wq));
        if (l16 == j) {
            tau_own = tau;
            scal_own = scal;
            beta_own = beta;
        }
        cplx g = cmul(cmul(scal, cconj(tau)), wq);
        g.x = l16 > j ? g.x : 0.0;
        g.y = l16 > j ? g.y : 0.0;
        // row j: v_j = 1 is (alpha - beta) scal
        {
            const bool rj = w == toff && lq == (j & 3);
            vb[0][j >> 2].x = rj ? amb.x : vb[0][j >> 2].x;
            vb[0][j >> 2].y = rj ? amb.y : vb[0][j >> 2].y;
        }
#pragma unroll
        for (int tt = 0; tt < FT; tt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                cplx v;
                if (FT <= FTW || tt == 0)
                    v = vb[tt][r];
                else {
                    // broadcast again (the empty asm: not kept from above, there are no registers for it)
                    asm volatile("" : "+v"(x.r[tt][r]), "+v"(x.i[tt][r]));
                    v = make_double2(row_bcast<j>(x.r[tt][r]), row_bcast<j>(x.i[tt][r]));
                }
                x.r[tt][r] = fma(-v.x, g.x, fma(v.y, g.y, x.r[tt][r]));
                x.i[tt][r] = fma(-v.x, g.y, fma(-v.y, g.x, x.i[tt][r]));
            }
    });
    // the reflectors in units of v_j = 1, beta on the diagonal
    if (l16 < b)
#pragma unroll
        for (int tt = 0; tt < FT; tt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = 4 * r + lq;
                const cplx v = cmul(make_double2(x.r[tt][r], x.i[tt][r]), scal_own);
                const bool below = tt > 0 || w > toff || (w == toff && row > l16), diag = tt == 0 && w == toff && row == l16;
                x.r[tt][r] = below ? v.x : diag ? beta_own : x.r[tt][r];
                x.i[tt][r] = below ? v.y : diag ? 0.0 : x.i[tt][r];
            }
}

// tau and T of the panel (wave 0, after the panel is stored: T's row takes the registers that held it)
template <int NW>
__device__ __forceinline__ void qr_tfactor(int b, cplx tau_own, GAS cplx *tau_out, GAS cplx *T, QrLds<NW> &L, int w, int lane)
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (w == 0 && lane < FPB) {
        // lane i builds row i of T: T(i, j) = -tau_j sum_{i <= q < j} T(i, q) S(q, j)
        const int i = lane;
        if (i < b) gst(tau_out + i, tau_own);
        cplx tr[FPB];
#pragma unroll
        for (int j = 0; j < FPB; j++) {
            tr[j] = make_double2(0.0, 0.0);
            if (j < b) {
                const cplx tj = make_double2(__shfl(tau_own.x, j, 16), __shfl(tau_own.y, j, 16));
                cplx a0 = make_double2(0.0, 0.0), a1 = a0;     // the two products of a term apart: half the chain
#pragma unroll
                for (int q = 0; q < j; q++) {
                    const cplx sq = L.S[j * FPB + q];
                    a0.x = fma(tr[q].x, sq.x, a0.x);
                    a0.y = fma(tr[q].x, sq.y, a0.y);
                    a1.x = fma(-tr[q].y, sq.y, a1.x);
                    a1.y = fma(tr[q].y, sq.x, a1.y);
                }
                const cplx v = cmul(make_double2(-tj.x, -tj.y), cadd(a0, a1));
                tr[j].x = j > i ? v.x : j == i ? tj.x : 0.0;
                tr[j].y = j > i ? v.y : j == i ? tj.y : 0.0;
            }
            gst(T + (j * FPB + i), tr[j]);
        }
    }
}

template <int NW, int FT>
__global__ void __launch_bounds__(64 * NW, 2)
k_qr_step(const DChain *chains, int sel, int k, int out_pt, int nc)
{
    __shared__ cplx red[NW * 256];
    __shared__ QrLds<NW> L;
    const DChain &c = chains[blockIdx.x];
    const int n = c.n, ncol = nc > 0 ? nc : n, kb = k + blockIdx.y, np = (ncol + FPB - 1) / FPB;
    if (kb >= np) return;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, lq = lane >> 4;
    const int k0 = FPB * max(k - 1, 0), m = n - k0, col = FPB * kb + l16, toff = k > 0 ? 1 : 0;
    GAS cplx *M = gp(chain_mat(c, sel, 0)), *A = M + k0;
    FBlk<FT> x;
    blk_load<NW>(x, A, n, m, col, ncol, w, lq, nullptr);
    if (k > 0)
        apply_panel<NW, true>(x, A + (size_t)k0 * n, n, m, min(FPB, m), gp(c.tblk) + (size_t)(k - 1) * FPB * FPB, 0, red,
                              w, lane, lq, l16);
    cplx tau_own = make_double2(0.0, 0.0);
    if (kb == k) qr_panel<NW>(x, min(FPB, ncol - FPB * k), toff, tau_own, L, w, lane, lq, l16);
#pragma unroll
    for (int tt = 0; tt < FT; tt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = 16 * (w + NW * tt) + 4 * r + lq;
            if (row < m && col < ncol) gst(A + ((size_t)row + (size_t)col * n), make_double2(x.r[tt][r], x.i[tt][r]));
        }
    if (kb == k)
        qr_tfactor<NW>(min(FPB, ncol - FPB * k), tau_own, gp(c.tau) + FPB * k, gp(c.tblk) + (size_t)k * FPB * FPB, L, w, lane);
    if (k == np - 1 && nc > 0) {
        // log|det R| and its negative diagonal entries
        __threadfence_block();
        __syncthreads();
        if (w == 0) {
            double rl = 0.0, neg = 0.0;
            for (int i = lane; i < ncol; i += 64) {
                const double r = gld(M + ((size_t)i + (size_t)i * n)).x;
                neg += r < 0.0 ? 1.0 : 0.0;
                rl += log(fabs(r));
            }
            rl = wave_sum_dpp(rl);
            neg = wave_sum_dpp(neg);
            if (lane == 0) {
                c.sc[SC_RLOG] = rl;
                c.sc[SC_RNEG] = neg;
            }
        }
    } else if (k == np - 1) {
        // log det Q = sum_i log(1 - tau_i 2 Re(tau_i) / |tau_i|^2), after the last panel
        __threadfence_block();
        __syncthreads();
        if (w == 0) {
            double sr = 0.0, si = 0.0;
            for (int i = lane; i < n; i += 64) {
                const cplx t = gld(gp(c.tau) + i);
                if (t.x != 0.0 || t.y != 0.0) {
                    const cplx q = cdiv(cscale(t, 2.0 * t.x), cmul(t, cconj(t)));
                    const cplx l = clog_(make_double2(1.0 - q.x, -q.y));
                    sr += l.x;
                    si += l.y;
                }
            }
            sr = wave_sum_dpp(sr);
            si = wave_sum_dpp(si);
            if (lane == 0) c.ldq[out_pt] = make_double2(sr, si);
        }
    }
}

// The columns 16 cb .. 16 cb + 15 of Q: the identity's columns through the panels cb .. 0 (the later ones
// leave them as they are).  The workgroups of a chain run on one XCD, which keeps the reflectors
// in its L2; the longest chains of panels start first.
template <int NW, int FT>
__global__ void __launch_bounds__(64 * NW, 2)
k_formq_cb(const DChain *chains, int nch, int ncb, int sel, int out_pt, int nc)
{
    __shared__ cplx red[2][NW * 256];
    const int bid = blockIdx.x, kb = bid >> 3, chain = (bid & 7) + 8 * (kb / ncb), cb = ncb - 1 - kb % ncb;
    if (chain >= nch) return;
    const DChain &c = chains[chain];
    const int n = c.n, ncol = nc > 0 ? nc : n;
    if (FPB * cb >= ncol) return;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, lq = lane >> 4;
    GAS cplx *A = gp(chain_mat(c, sel, 0)), *Q = gp(c.U + (size_t)n * n * out_pt);
    FBlk<FT> x;
#pragma unroll
    for (int tt = 0; tt < FT; tt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            x.r[tt][r] = w + NW * tt == cb && 4 * r + lq == l16 ? 1.0 : 0.0;
            x.i[tt][r] = 0.0;
        }
    for (int p = cb; p >= 0; p--) {
        const int k0 = FPB * p;
        apply_panel<NW, false>(x, A + ((size_t)k0 + (size_t)k0 * n), n, n - k0, min(FPB, ncol - k0),
                               gp(c.tblk) + (size_t)p * FPB * FPB, p, red[p & 1], w, lane, lq, l16);
    }
    const int col = FPB * cb + l16;
    // a tall matrix's first column of Q takes the sign of det R (s_zgeQR_pqmc)
    const bool flip = nc > 0 && col == 0 && ((int)c.sc[SC_RNEG] & 1);
#pragma unroll
    for (int tt = 0; tt < FT; tt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = 16 * (w + NW * tt) + 4 * r + lq;
            if (row < n && col < ncol)
                gst(Q + ((size_t)row + (size_t)col * n), make_double2(flip ? -x.r[tt][r] : x.r[tt][r], flip ? -x.i[tt][r] : x.i[tt][r]));
        }
}

template <int NW>
struct LuLds {
    cplx row[2][NW][16];
    double v[2][NW];
    int p[2][NW], prow[FPB];
};

// the lane's entry e (0 .. 4 FTW - 1) to *dst by a binary tree of uniform branches; the empty asm keeps
// each leaf a branch target of its own (merged, they index the registers through private memory)
template <int LO, int HI>
__device__ __forceinline__ void blk_pick(const FBlk<FTW> &x, int e, cplx *dst)
{
    if constexpr (HI - LO == 1) {
        *dst = make_double2(x.r[LO >> 2][LO & 3], x.i[LO >> 2][LO & 3]);
        asm volatile("" ::: "memory");
    } else {
        constexpr int MID = (LO + HI) / 2;
        if (e < MID)
            blk_pick<LO, MID>(x, e, dst);
        else
            blk_pick<MID, HI>(x, e, dst);
    }
}

// LU of the panel in x (b columns, m rows from tile toff) without moving rows.  act: bit e is set while
// the lane's row of entry e is still to be eliminated.  Per column every wave finds its largest |Re| + |Im|
// among those rows (the first of equal ones) and publishes it with that row's entries; behind the one
// barrier every lane takes the best wave's row as the pivot row.  A column stays unscaled until the
// end (its lanes keep 1 / pivot and the rows below).  L.prow: the pivot rows.  The interchanges displace
// only the rows 0 .. 15: lane i < 16 of every row group keeps where = the place of row i and top = the row
// at place i.
template <int NW>
__device__ __forceinline__ void lu_panel(FBlk<FTW> &x, int &act, int b, int toff, GAS int32_t *piv, int k0, double *info, LuLds<NW> &L,
                                         int &where, int w, int lane, int lq, int l16)
{
    int top = l16, below = 0;
    cplx pinv_own = make_double2(1.0, 0.0);
    where = l16;
    cols16([&](auto jc) {
        constexpr int j = decltype(jc)::value, par = j & 1;
        if (j >= b) return;
        double bv = -1.0;
        int be = 0;
#pragma unroll
        for (int e = 0; e < 4 * FTW; e++) {
            double v = fabs(x.r[e >> 2][e & 3]) + fabs(x.i[e >> 2][e & 3]);
            v = act >> e & 1 ? v : -1.0;
            be = v > bv ? e : be;
            bv = v > bv ? v : bv;
        }
        // as a row of the panel: 16 (w + NW tt - toff) + 4 r + lq
        int bp = 16 * (w + NW * (be >> 2) - toff) + 4 * (be & 3) + lq;
        auto take = [&](double v2, int p2) {
            const bool t = v2 > bv || (v2 == bv && p2 < bp);
            bv = t ? v2 : bv;
            bp = t ? p2 : bp;
        };
        take(swap16_d(bv), swap16_i(bp));
        take(swap32_d(bv), swap32_i(bp));
        // column j's candidate (lane j of any row group), the same in every lane
        const double wv = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(bv), j),
                                           __builtin_amdgcn_readlane(__double2loint(bv), j));
        const int wp = __builtin_amdgcn_readlane(bp, j);
        // its entry: tile (wp/16 + toff - w) / NW, element (wp % 16) / 4 of the lanes l/16 = wp % 4
        const int we = ((((wp >> 4) + toff - w) / NW) << 2) + ((wp & 15) >> 2);
        if (lq == (wp & 3)) blk_pick<0, 4 * FTW>(x, we, &L.row[par][w][l16]);
        if (lane == 0) {
            L.v[par][w] = wv;
            L.p[par][w] = wp;
        }
        __syncthreads();
        double gv = L.v[par][0];
        int gr = L.p[par][0], gw = 0;
#pragma unroll
        for (int q = 1; q < NW; q++) {
            const double v2 = L.v[par][q];
            const int p2 = L.p[par][q];
            const bool t = v2 > gv || (v2 == gv && p2 < gr);
            gv = t ? v2 : gv;
            gr = t ? p2 : gr;
            gw = t ? q : gw;
        }
        gr = __builtin_amdgcn_readfirstlane(gr);
        gw = __builtin_amdgcn_readfirstlane(gw);
        if (!(gv >= 0.0)) gr = __builtin_amdgcn_readlane(top, j);   // no comparable entry (NaN): the row in place
        // the interchange of places j and gpos
        const int gpos = gr < 16 ? __builtin_amdgcn_readlane(where, gr & 15) : gr, tj = __builtin_amdgcn_readlane(top, j);
        where = l16 == tj ? gpos : where;
        where = l16 == gr ? j : where;
        top = l16 == gpos ? tj : top;
        if (threadIdx.x == 0) {
            piv[j] = k0 + gpos;
            L.prow[j] = gr;
        }
        // the pivot row leaves the active ones
        const int ge = ((((gr >> 4) + toff - w) / NW) << 2) + ((gr & 15) >> 2);
        if ((gr >> 4) + toff >= w && ((gr >> 4) + toff - w) % NW == 0 && lq == (gr & 3))
            act &= ~(1 << ge);
        cplx u = L.row[par][gw][l16];
        const cplx pv = make_double2(row_bcast<j>(u.x), row_bcast<j>(u.y));
        const bool skip = !(gv > 0.0);
        if (gv == 0.0 && threadIdx.x == 0 && *info == 0.0) *info = (double)(k0 + j + 1);
        cplx pinv = cinv_s(pv);
        pinv.x = skip ? 0.0 : pinv.x;
        pinv.y = skip ? 0.0 : pinv.y;
        if (l16 == j) {
            pinv_own.x = skip ? 1.0 : pinv.x;
            pinv_own.y = pinv.y;
            below = act;
        }
        // the rows still active -= (their column j entry / pivot) u; f = u / pivot
        u.x = l16 > j ? u.x : 0.0;
        u.y = l16 > j ? u.y : 0.0;
        const cplx f = cmul(u, pinv);
#pragma unroll
        for (int e = 0; e < 4 * FTW; e++) {
            const double cx = row_bcast<j>(x.r[e >> 2][e & 3]), cy = row_bcast<j>(x.i[e >> 2][e & 3]);
            const bool in = act >> e & 1;
            const double lx = in ? cx : 0.0, ly = in ? cy : 0.0;
            x.r[e >> 2][e & 3] = fma(-lx, f.x, fma(ly, f.y, x.r[e >> 2][e & 3]));
            x.i[e >> 2][e & 3] = fma(-lx, f.y, fma(-ly, f.x, x.i[e >> 2][e & 3]));
        }
    });
    if (l16 < b)
#pragma unroll
        for (int e = 0; e < 4 * FTW; e++) {
            const cplx l = cmul(make_double2(x.r[e >> 2][e & 3], x.i[e >> 2][e & 3]), pinv_own);
            const bool in = below >> e & 1;
            x.r[e >> 2][e & 3] = in ? l.x : x.r[e >> 2][e & 3];
            x.i[e >> 2][e & 3] = in ? l.y : x.i[e >> 2][e & 3];
        }
}

// Launch k = 0 .. np (np panels) on W3.  Panel k leaves in lup + k FLMAX the map of its interchanges: the
// row (relative to row 16 k) that comes to each place from row 16 k on.  Launch np brings the columns
// left of each panel into the final row order and sums the log determinant (s_inv_logdet_lu_z: Im
// folded into (-pi, pi]) to the scalar slot zslot, if not negative; fresh clears the zero-pivot slot first; lperm is the row order of all interchanges (row i of P X is row lperm[i] of X).
template <int NW>
__global__ void __launch_bounds__(64 * NW, 2)
k_lu_step(const DChain *chains, int k, int zslot, int fresh)
{
    __shared__ cplx Xp[256], D11[256];
    __shared__ LuLds<NW> L;
    __shared__ int ord[64 * NW];
    const DChain &c = chains[blockIdx.x];
    const int n = c.n, np = (n + FPB - 1) / FPB, kb = (k < np ? k : 0) + blockIdx.y;
    if (k > np || kb >= np) return;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, lq = lane >> 4;
    GAS cplx *M = gp(c.W3);
    GAS int32_t *lup = gp(c.lup);
    const int col = FPB * kb + l16;
    FBlk<FTW> x;
    if (k == np) {
        if (kb == np - 1) {
            if (w == 0) {
                double lr = 0.0, li = 0.0;
                for (int i = lane; i < n; i += 64) {
                    cplx d = gld(M + ((size_t)i + (size_t)i * n));
                    if (c.piv[i] != i) d = make_double2(-d.x, -d.y);
                    const cplx l = clog_(d);
                    lr += l.x;
                    li += l.y;
                }
                lr = wave_sum_dpp(lr);
                li = wave_sum_dpp(li);
                if (lane == 0 && zslot >= 0) {
                    const double k2 = round(li / 2.0 / M_PI);
                    c.sc[zslot] = lr;
                    c.sc[zslot + 1] = li - 2.0 * M_PI * k2;
                }
            }
            return;
        }
        // the block's rows below its own panel through the maps of the later panels, last one first
        const int r0 = FPB * (kb + 1), m = n - r0;
        for (int i = threadIdx.x; i < m; i += 64 * NW) {
            int q = r0 + i;
            for (int p = np - 1; p > kb; p--)
                if (q >= FPB * p) q = FPB * p + lup[(size_t)p * FLMAX + q - FPB * p];
            ord[i] = q - r0;
        }
        __syncthreads();
        GAS cplx *A = M + r0;
        const size_t cc = (size_t)col * n;
#pragma unroll
        for (int tt = 0; tt < FTW; tt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const cplx v = gld(A + ((size_t)ord[min(16 * (w + NW * tt) + 4 * r + lq, m - 1)] + cc));
                x.r[tt][r] = v.x;
                x.i[tt][r] = v.y;
            }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
#pragma unroll
        for (int tt = 0; tt < FTW; tt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = 16 * (w + NW * tt) + 4 * r + lq;
                if (row < m) gst(A + ((size_t)row + cc), make_double2(x.r[tt][r], x.i[tt][r]));
            }
        return;
    }
    const int k0 = FPB * max(k - 1, 0), m = n - k0, toff = k > 0 ? 1 : 0;
    GAS cplx *A = M + k0;
    blk_load<NW>(x, A, n, m, col, n, w, lq, k > 0 ? lup + (size_t)(k - 1) * FLMAX : (const GAS int32_t *)nullptr);
    if (k > 0) {
        GAS cplx *V = A + (size_t)k0 * n;
        // U12 = L11^-1 X (rows of tile 0, wave 0), column by column of L11
        if (w == 0) {
#pragma unroll
            for (int e4 = 0; e4 < 4; e4++) {
                const int e = lane + 64 * e4;
                D11[e] = gld(V + ((size_t)(e & 15) + (size_t)(e >> 4) * n));     // D11[b * 16 + a] = L(a, b)
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
            for (int q = 0; q < 15; q++) {
                const int src = l16 + 16 * (q & 3);
                const double vr = __shfl(x.r[0][q >> 2], src, 64), vi = __shfl(x.i[0][q >> 2], src, 64);
#pragma unroll
                for (int r = q >> 2; r < 4; r++) {
                    const int a = 4 * r + lq;
                    const cplx l = D11[q * 16 + a];
                    const double lx = a > q ? l.x : 0.0, ly = a > q ? l.y : 0.0;
                    x.r[0][r] = fma(-lx, vr, fma(ly, vi, x.r[0][r]));
                    x.i[0][r] = fma(-lx, vi, fma(-ly, vr, x.i[0][r]));
                }
            }
#pragma unroll
            for (int r = 0; r < 4; r++) Xp[(4 * r + lq) * 16 + l16] = make_double2(x.r[0][r], x.i[0][r]);
        }
        // every load of this block has landed before any wave stores a row
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        cplx bx[4];
#pragma unroll
        for (int s = 0; s < 4; s++) bx[s] = Xp[(4 * s + lq) * 16 + l16];
#pragma unroll
        for (int tt = 0; tt < FTW; tt++) {
            const int rt = w + NW * tt;
            if (rt > 0 && 16 * rt < m) {
                cplx a[4];
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    const int row = 16 * rt + l16;
                    const cplx v = gld(V + ((size_t)min(row, m - 1) + (size_t)(4 * s + lq) * n));
                    a[s].x = row < m ? v.x : 0.0;
                    a[s].y = row < m ? v.y : 0.0;
                }
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    x.r[tt] = mfma(-a[s].x, bx[s].x, x.r[tt]);
                    x.i[tt] = mfma(-a[s].x, bx[s].y, x.i[tt]);
                    x.r[tt] = mfma(a[s].y, bx[s].y, x.r[tt]);
                    x.i[tt] = mfma(-a[s].y, bx[s].x, x.i[tt]);
                }
            }
        }
    }
    if (kb != k) {
#pragma unroll
        for (int tt = 0; tt < FTW; tt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = 16 * (w + NW * tt) + 4 * r + lq;
                if (row < m && col < n) gst(A + ((size_t)row + (size_t)col * n), make_double2(x.r[tt][r], x.i[tt][r]));
            }
        return;
    }
    // panel k
    const int q0 = FPB * k, mp = n - q0, b = min(FPB, mp);
    int act = 0;
#pragma unroll
    for (int e = 0; e < 4 * FTW; e++) {
        const int row = 16 * (w + NW * (e >> 2) - toff) + 4 * (e & 3) + lq;
        act |= row >= 0 && row < mp ? 1 << e : 0;
    }
    if (threadIdx.x == 0 && k == 0 && fresh) c.sc[SC_INFO] = 0.0;
    // the row order before this panel, loaded before any of it is replaced
    int lp[4 * FTW];
#pragma unroll
    for (int e = 0; e < 4 * FTW; e++) {
        const int row = min(max(16 * (w + NW * (e >> 2) - toff) + 4 * (e & 3) + lq, 0), mp - 1);
        lp[e] = k > 0 ? c.lperm[q0 + row] : row;
    }
    for (int i = FPB + threadIdx.x; i < mp; i += 64 * NW) ord[i] = i;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int where;
    lu_panel<NW>(x, act, b, toff, gp(c.piv) + q0, q0, c.sc + SC_INFO, L, where, w, lane, lq, l16);
    __syncthreads();
    // the place of every row: rows 0 .. 15 where the interchanges put them (every wave's lanes hold the same),
    // a pivot row from below at its step, every other row where it was
    if (w == 0 && lane < FPB) {
        ord[lane] = where;
        if (lane < b && L.prow[lane] >= FPB) ord[L.prow[lane]] = lane;
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4 * FTW; e++) {
        const int src = 16 * (w + NW * (e >> 2) - toff) + 4 * (e & 3) + lq;
        const int place = src < 0 ? src : ord[min(src, mp - 1)];     // rows above the panel: its U block
        if (src < mp && col < n) {
            gst(M + ((size_t)(q0 + place) + (size_t)col * n), make_double2(x.r[e >> 2][e & 3], x.i[e >> 2][e & 3]));
            if (src >= 0 && l16 == 0) {
                lup[(size_t)k * FLMAX + place] = src;
                c.lperm[q0 + place] = lp[e];
            }
        }
    }
}

#define QR(NW, FT)                                                                          \
    template __global__ void k_qr_step<NW, FT>(const DChain *, int, int, int, int);          \
    template __global__ void k_formq_cb<NW, FT>(const DChain *, int, int, int, int, int);
QR(4, FTW)
QR(8, FTW)
QR(8, 2 * FTW)
template __global__ void k_lu_step<4>(const DChain *, int, int, int);
template __global__ void k_lu_step<8>(const DChain *, int, int, int);
