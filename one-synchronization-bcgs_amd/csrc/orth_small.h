// The small-matrix steps between passes (FP64, one workgroup of nt threads,
// nt a multiple of 64 and at least 256): Pythagorean Gram, Cholesky factors
// with their solve blocks, lag correction, R assembly and the next pass's
// coefficients.  Run by k_small on its own or by the last workgroup of
// k_reduce_small.
//
// What bounds a step is its dependent chain, not its arithmetic (< 1 Mflop):
// memory round trips (about 1 us each for data another workgroup just
// wrote), the division of every Cholesky pivot, workgroup barriers, and the
// fetch of its own code, which each launch runs once on whatever CU holds the
// last workgroup (a form of these steps with the factorizations and solves
// unrolled in registers took 33 us where this one takes 23 us, both with the
// launch and the reduction: closing a 10-column block with 130 columns before
// it; pivots by one thread with every intermediate in global memory took
// 65 us).  So:
//   * everything a step reads is requested in one round: the rows below the
//     prefix go to LDS while the Gram of the prefix rows [Y S] (all of Y^T Y,
//     Y^T S and S^T S that the step needs) runs on FP64 MFMA, 16 x 16 tiles
//     with the prefix rows split over the waves;
//   * closing one block and opening the next is one Cholesky factorization:
//     [[Om, S_bot], [0, Sigma_n]] is the upper factor of
//     [[H, W], [W^T, G_n]], H and G_n the Pythagorean Grams and W the lagged
//     projection.  One wave eliminates it (rolled loops, entries in
//     registers, pivot rows through LDS), the others assemble R meanwhile;
//   * the c x s products for R and the coefficients are MFMA tiles.
//
// W: 16 or 32, at least the block widths.
#pragma once

#include <hip/hip_runtime.h>

#include "orth_device.h"
#include "orth_kernels.h"

namespace orth {

// LDS layout (doubles): the 2W x 2W matrix M of the step (row-major, ld L; a
// block's own columns at 0, the next block's at W), the reciprocal pivots,
// the Gram partials (at most kItems tiles of 16 x 16; their space is reused
// for Z2 and the CholQR products, ld LZ), the breakdown pivots.
template <int W>
struct SmallLay {
    static constexpr int LW = W == 16 ? 4 : 5;
    static constexpr int L = 2 * W + 2, LZ = W + 2;
    static constexpr int kItems = W == 16 ? 16 : 10;
    static constexpr int M = 0, RC = 2 * W * L, Z = RC + 2 * W;
    static constexpr int Info = Z + kItems * 256, Size = Info + 2;
    static_assert(kItems * 256 >= 2 * W * LZ, "the CholQR products reuse the Gram partials' space");
};
// Doubles of LDS a small step needs.
template <int W>
constexpr int small_lds()
{
    return SmallLay<W>::Size;
}

static __device__ __forceinline__ void wave_fence()
{
    // A wave's LDS accesses execute in order; the fence stops the compiler
    // from moving or forwarding them.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// Gram of the prefix: tiles [p][q] of [Y S]^T [Y S] over rows [0, c) of P
// (Y = columns [0, w0), S = columns [w0, w0 + w1)), Y and S padded to whole
// 16-column tiles.  Pairs p <= q in row-major order, without the S-S pairs
// when !ss; each pair's rows are split into KS = kItems / pairs slices, and
// item (pair, slice) leaves its 16 x 16 partial tile at
// part[256 (pair KS + slice)].
template <int W>
struct GramPlan {
    int nY, nT, np, KS;
    __device__ __forceinline__ GramPlan(int w0, int w1, bool ss)
    {
        nY = (w0 + 15) >> 4;
        nT = nY + ((w1 + 15) >> 4);
        const int lim = ss ? nT : nY;
        np = 0;
        for (int p = 0; p < lim; p++) np += nT - p;
        KS = SmallLay<W>::kItems / np;
    }
    __device__ __forceinline__ void pair(int i, int *p, int *q) const
    {
        int a = 0;
        while (i >= nT - a) {
            i -= nT - a;
            a++;
        }
        *p = a;
        *q = a + i;
    }
};

template <int W>
static __device__ __forceinline__ void d_gram(int nt, const GramPlan<W> &gp, int c, int w0, int w1,
                                              const double *P, int64_t na, double *part)
{
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nblk = (c + 15) >> 4;  // 16-row blocks of the prefix
    for (int it = wave; it < gp.np * gp.KS; it += nt >> 6) {
        int p, q;
        gp.pair(it / gp.KS, &p, &q);
        const int ks = it % gp.KS;
        // Column of this lane in tile t, or -1 past the block.
        auto col = [&](int t) {
            const int j = 16 * (t < gp.nY ? t : t - gp.nY) + li;
            return t < gp.nY ? (j < w0 ? j : -1) : (j < w1 ? w0 + j : -1);
        };
        const int cp = col(p), cq = col(q);
        const double *Pp = P + (int64_t)max(cp, 0) * na, *Pq = P + (int64_t)max(cq, 0) * na;
        dbl4 z = dbl4{0.0, 0.0, 0.0, 0.0};
        const int b1 = nblk * (ks + 1) / gp.KS, re = min(c, 16 * b1);
        // A lane takes four consecutive rows of its column per 16-row block
        // (any assignment of rows to k-steps gives the same sum); two blocks
        // of loads in flight.
        for (int b = nblk * ks / gp.KS; b < b1; b += 2) {
            double x[8], y[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int r = 16 * (b + (e >> 2)) + 4 * lk + (e & 3);
                x[e] = r < re && cp >= 0 ? Pp[r] : 0.0;
                y[e] = r < re && cq >= 0 ? Pq[r] : 0.0;
            }
#pragma unroll
            for (int e = 0; e < 8; e++)
                z = __builtin_amdgcn_mfma_f64_16x16x4f64(x[e], y[e], z, 0, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < 4; v++) part[256 * it + (lk + 4 * v) * 16 + li] = z[v];
    }
}

// One wave: M(r0 + i, c0 + j) -= sum_{l < k} M(l, r0 + i) M(l, c0 + j) for
// i < nr, j < nc (LDS, ld L; rows past k read as zero), 16 x 16 MFMA tiles;
// with tri only the tiles on or right of the diagonal.
template <int W>
static __device__ __forceinline__ void wave_syrk(int k, int r0, int nr, int c0, int nc, bool tri,
                                                 double *M)
{
    constexpr int L = SmallLay<W>::L;
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    for (int p = 0; p < nr; p += 16)
        for (int q = tri ? p : 0; q < nc; q += 16) {
            dbl4 z = dbl4{0.0, 0.0, 0.0, 0.0};
            for (int l0 = 0; l0 < k; l0 += 4) {
                const double *Ml = M + (l0 + lk) * L;
                const double x = l0 + lk < k ? Ml[r0 + p + li] : 0.0;
                const double y = l0 + lk < k ? Ml[c0 + q + li] : 0.0;
                z = __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, z, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = p + lk + 4 * v, jj = q + li;
                if (i < nr && jj < nc) M[(r0 + i) * L + c0 + jj] -= z[v];
            }
        }
}

// One wave: rows [0, w) and columns [0, nc) of M (LDS, ld L; nc <= 2W) <- the
// rows of the upper factor U of M's leading w x w block, U^T U = M, with
// U^{-T} M in the columns past w; strict lower zeroed; rc[i] = 1 / U(i, i).
// Sixteen rows at a time (the rows above are subtracted on MFMA first):
// right-looking elimination, a lane keeps every RG-th row of one column in
// registers, the pivot row goes through LDS, and the only division on the
// chain is the pivot's reciprocal (the square roots scale the rows at the
// end); a pivot whose reciprocal would leave the normal range goes through its
// square root instead.  A pivot that is not positive makes everything after
// it NaN.
// *info: 0 or the 1-based first such pivot.
template <int W>
static __device__ __forceinline__ void wave_chol(int w, int nc, double *M, double *rc, int *info)
{
    constexpr int L = SmallLay<W>::L, RG = 32 / W, NQ = 16 / RG;
    const int lane = threadIdx.x & 63, j = lane & (2 * W - 1), h = lane / (2 * W);
    const bool act = j < nc;
    int bad = 0;
    for (int b0 = 0; b0 < w; b0 += 16) {
        const int wb = min(16, w - b0);
        if (b0 > 0) {
            wave_syrk<W>(b0, b0, wb, b0, nc - b0, false, M);
            wave_fence();
        }
        double *Mb = M + b0 * L;
        double m[NQ];
#pragma unroll
        for (int q = 0; q < NQ; q++) m[q] = act && RG * q + h < wb ? Mb[(RG * q + h) * L + j] : 0.0;
        for (int k = 0; k < wb; k++) {
            const double *Mk = Mb + k * L;
            const double d = Mk[b0 + k], mk = act ? Mk[j] : 0.0;
            double a[NQ];
#pragma unroll
            for (int q = 0; q < NQ; q++) a[q] = Mk[b0 + RG * q + h];
            double r = 1.0 / d, x = mk;
            // One scalar comparison beside the chain: 2^-1000 <= d < 2^1000.
            const uint32_t hi = __builtin_amdgcn_readfirstlane(__double2hiint(d));
            if (__builtin_expect(hi - (23u << 20) >= 2000u << 20, 0)) {
                if (d > 0.0) {
                    r = 1.0 / sqrt(d);
                    x = mk * r;
                } else {
                    r = __builtin_nan("");
                    if (bad == 0) bad = b0 + k + 1;
                }
            }
#pragma unroll
            for (int q = 0; q < NQ; q++)
                if (RG * q + h > k) m[q] = fma(-(a[q] * r), x, m[q]);
#pragma unroll
            for (int q = 0; q < NQ; q++)
                if (act && RG * q + h < wb) Mb[(RG * q + h) * L + j] = m[q];
            wave_fence();
        }
        const double u = lane < wb ? sqrt(Mb[lane * L + b0 + lane]) : 1.0;
        if (lane < wb) rc[b0 + lane] = 1.0 / u;
        wave_fence();
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const int i = RG * q + h;
            if (act && i < wb) Mb[i * L + j] = j < b0 + i ? 0.0 : m[q] * rc[b0 + i];
        }
        wave_fence();
        if (lane < wb) Mb[lane * L + b0 + lane] = u;
        wave_fence();
    }
    if (lane == 0) *info = bad;
}

// One wave: Z (w0 x w1, ld LZ) = Om^{-1} S_bot, Om at M(0, 0) and S_bot at
// M(0, W): back substitution, right-looking, rows of Z through LDS.
template <int W>
static __device__ __forceinline__ void wave_solve_z2(int w0, int w1, const double *M, double *Z)
{
    constexpr int L = SmallLay<W>::L, LZ = SmallLay<W>::LZ, RG = 64 / W, NQ = W / RG;
    const int lane = threadIdx.x & 63, j = lane & (W - 1), h = lane / W;
    const bool act = j < w1;
    double m[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const int l = RG * q + h;
        m[q] = act && l < w0 ? M[l * L + W + j] : 0.0;
        Z[l * LZ + j] = m[q];
    }
    wave_fence();
    for (int i = w0 - 1; i >= 0; i--) {
        const double x = Z[i * LZ + j] / M[i * (L + 1)];
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const int l = RG * q + h;
            const double u = M[min(l, i) * L + i];
            m[q] = l < i ? fma(-u, x, m[q]) : l == i ? x : m[q];
        }
        // Row i's owner stores its solution, the others their updated rows.
#pragma unroll
        for (int q = 0; q < NQ; q++) Z[(RG * q + h) * LZ + j] = m[q];
        wave_fence();
    }
}

// Threads t of n: the factor slot T (layout in orth_kernels.h) of the w x w
// factor M in LDS (ld L, reciprocal pivots rc): the factor, the reciprocals
// and the row blocks of the blocked solve, whose row D_b(k, :) of the
// inverted 4 x 4 diagonal block each thread forms for itself:
// D(k,k) = 1/u(k,k), D(k,j) = -(sum_{i=k}^{j-1} D(k,i) u(i,j)) / u(j,j).
// Entries past W keep the zeros the call started with.  p: the first bad pivot
// (w: none); the row blocks then solve for the columns before it and leave NaN
// in the others (see orth_kernels.h).
template <int W>
static __device__ __forceinline__ void d_write_slot(int t, int n, int w, int p, const double *M,
                                                    const double *rc, double *T)
{
    constexpr int L = SmallLay<W>::L, LW = SmallLay<W>::LW;
    for (int e = t; e < W * W; e += n) {
        const int i = e >> LW, c = e & (W - 1), o = i & ~3;
        const bool in = i < w && c < w;
        T[i + c * kLdT] = in && i <= c ? M[i * L + c] : 0.0;
        if (c == 0) T[kSlotRecip + i] = i < w ? rc[i] : 0.0;
        double d[4], v = 0.0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < j; k++) s = fma(d[k], M[(o + k) * L + o + j], s);
            // Zero left of the diagonal (k < i - o) and past the factor.
            d[j] = o + j < i || o + j >= w ? 0.0 : o + j == i ? rc[i] : -s * rc[o + j];
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
            v = c >= o + 4 ? (o + j < w ? fma(-d[j], M[(o + j) * L + c], v) : v) : c == o + j ? d[j] : v;
        if (p < w && (i >= p || c >= p))
            v = c >= p && o == slot_last(c, w) ? __builtin_nan("") : 0.0;
        T[kSlotW + o * kLdT + (i & 3) * kLdT + c] = in ? v : 0.0;
    }
}

// Threads t of n: C = A B for upper-triangular A (w x w, LDS, row-major ld
// la) and B (slot layout, ld kLdT); entry (i, j) of C at C[i si + j sj],
// strict lower zero.
template <int W>
static __device__ __forceinline__ void d_trmm(int t, int n, int w, const double *A, int la,
                                              const double *B, double *C, int64_t si, int64_t sj)
{
    for (int e = t; e < W * W; e += n) {
        const int i = e & (W - 1), j = e >> SmallLay<W>::LW;
        if (i >= w || j >= w) continue;
        double s = 0.0;
        for (int l = i; l <= j; l++) s = fma(A[i * la + l], B[l + j * kLdT], s);
        C[i * si + j * sj] = i <= j ? s : 0.0;
    }
}

// Rows of a 16-row tile in the MFMA layouts used below: A-operand lane li
// holds row trow(li), so that result value v of lane lk is row 4 lk + v (four
// consecutive rows per lane).
static __device__ __forceinline__ int trow(int li) { return 4 * (li & 3) + (li >> 2); }

// Waves [wlo, nt / 64): the prefix rows of R, in 16 x 16 tiles: R(0:c, 0:w0)
// at Rb takes Y (mode 0: =, 1: += Y, 2: += Y Sigma, Sigma the upper factor in
// slot layout) and R(0:c, w0:w0+w1) = S.
template <int W>
static __device__ __forceinline__ void d_r_rows(int nt, int wlo, int mode, int c, int w0, int w1,
                                                const double *P, int64_t na, const double *Sig,
                                                double *Rb, int64_t ldR)
{
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nY = (w0 + 15) >> 4, nT = nY + ((w1 + 15) >> 4), ntask = ((c + 15) >> 4) * nT;
    for (int t = wave - wlo; t < ntask; t += (nt >> 6) - wlo) {
        const int r0 = 16 * (t / nT), tn = t % nT;
        const bool y = tn < nY;
        const int jl = 16 * (y ? tn : tn - nY) + li;  // column within Y or S
        const bool jok = jl < (y ? w0 : w1);
        const int col = y ? jl : w0 + jl;
        dbl4 z = dbl4{0.0, 0.0, 0.0, 0.0};
        if (y && mode == 2) {
            const int rr = r0 + trow(li);
            for (int l0 = 0; l0 < w0; l0 += 4) {
                const int l = l0 + lk;
                const double x = rr < c && l < w0 ? P[rr + (int64_t)l * na] : 0.0;
                const double s = l <= jl && jok ? Sig[l + jl * kLdT] : 0.0;
                z = __builtin_amdgcn_mfma_f64_16x16x4f64(x, s, z, 0, 0, 0);
            }
        }
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = r0 + 4 * lk + v;
            if (row < c && jok) {
                double *R = Rb + row + (int64_t)col * ldR;
                const double x = y && mode == 2 ? z[v] : P[row + (int64_t)col * na];
                *R = y && mode > 0 ? *R + x : x;
            }
        }
    }
}

// Every wave: coefficients of the next fused pass, row-major C[k][n] (ld n1;
// W = 32: in the order of wpass_cidx) for k < roundup4(k1), in 16 x 16 tiles: columns [0, w0) are Y over rows
// [0, c), zero below; columns [S, S + w1) are S_top over rows [0, c) (with
// sub: S_top - Y Z) and the w0 x w1 block Z in LDS (ld lz) over rows
// [c, c + w0); everything else is zero.
template <int W>
static __device__ __forceinline__ void d_emit(int nt, double *C, int n1, int S, int k1, int c,
                                              int w0, int w1, const double *P, int64_t na,
                                              const double *Z, int lz, bool sub)
{
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int k1p = (k1 + 3) & ~3, nN = n1 >> 4, ntask = ((k1p + 15) >> 4) * nN;
    for (int t = wave; t < ntask; t += nt >> 6) {
        const int r0 = 16 * (t / nN), n = 16 * (t % nN) + li;
        const bool g1 = n >= S;
        const int j = g1 ? n - S : n, col = g1 ? w0 + j : j;
        const bool jok = j < (g1 ? w1 : w0);
        dbl4 z = dbl4{0.0, 0.0, 0.0, 0.0};
        if (sub && 16 * (t % nN) + 15 >= S) {
            const int rr = r0 + trow(li);
            for (int l0 = 0; l0 < w0; l0 += 4) {
                const int l = l0 + lk;
                const double x = rr < c && l < w0 ? P[rr + (int64_t)l * na] : 0.0;
                const double s = g1 && jok && l < w0 ? Z[l * lz + j] : 0.0;
                z = __builtin_amdgcn_mfma_f64_16x16x4f64(x, s, z, 0, 0, 0);
            }
        }
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int k = r0 + 4 * lk + v;
            if (k < k1p) {
                double x = 0.0;
                if (jok && k < c) x = P[k + (int64_t)col * na] - z[v];
                if (jok && g1 && k >= c && k < c + w0) x = Z[(k - c) * lz + j];
                C[W == 32 ? wpass_cidx(k, n) : k * n1 + n] = x;
            }
        }
    }
}

static __device__ __forceinline__ void note_info(int *status, int blk, int info)
{
    if (info != 0 && status[0] == 0) {
        status[0] = blk + 1;
        status[1] = info;
    }
}

// One small step (SmallArgs::op); lds: small_lds<W>() doubles of LDS.
//   OP_OPEN_PYTH   G -= S^T S; R(0:c, b) = S; Sigma = chol(G) (SRC/orth.c:115-119)
//   OP_PIPI1       the same (SRC/orth.c:425-429)
//   OP_CLOSE_OPEN  SRC/orth.c:134-171, :200-215 (:356-360 with F_1S)
//   OP_PIPI2       SRC/orth.c:440-455
//   OP_PLAIN_S     R(0:c, b) = S; OP_I2_W R(0:c, b) += W Sigma
//   OP_CQR1..3     the steps of the shifted CholQR3
template <int W>
static __device__ __forceinline__ void small_step(int nt, const SmallArgs &a, double *lds)
{
    using Lay = SmallLay<W>;
    constexpr int L = Lay::L, LW = Lay::LW, LZ = Lay::LZ;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int op = a.op, c = a.c, wb = a.wb, wn = a.wn, na = a.na;
    double *P = a.P;
    double *Rb = a.R + (int64_t)c * a.ldR;  // R(:, block b)
    double *M = lds + Lay::M, *rc = lds + Lay::RC, *Z = lds + Lay::Z;
    int *info = (int *)(lds + Lay::Info);
    const bool qr = op >= OP_CQR1 && op <= OP_CQR3;
    const bool close = op == OP_CLOSE_OPEN || op == OP_PIPI2;
    const bool pyth = wn > 0 && (a.flags & F_PYTH_NEXT);
    const int mode = op == OP_I2_W || (close && !(a.flags & F_1S)) ? 2 : close ? 1 : 0;

    if (op == OP_PLAIN_S || op == OP_I2_W) {
        if (a.Cout) d_emit<W>(nt, a.Cout, a.n1, a.S, c, c, wb, 0, P, na, Z, LZ, false);
        d_r_rows<W>(nt, 0, mode, c, wb, 0, P, na, a.Sig, Rb, a.ldR);
        return;
    }

    // The rows of P below the prefix go to M: G of this block at (0, 0) (the
    // whole of P for a CholQR step), the next block's projection on it at
    // (0, W) and its Gram at (W, W); upper triangles of the Grams, a shift
    // on their diagonals.
    const int bot = qr ? 0 : c;
    double *Pn = P + (int64_t)wb * na;
    double sh0 = 0.0, sh1 = 0.0;
    if (op == OP_CQR1 || a.pshift != 0.0) {
        double t0 = 0.0, t1 = 0.0;
        for (int i = 0; i < wb; i++) t0 += P[bot + i + (int64_t)i * na];
        if (pyth)
            for (int i = 0; i < wn; i++) t1 += Pn[c + wb + i + (int64_t)i * na];
        const double u = 1.1102230246251565e-16;
        // Pythagorean steps: pshift u tr(G).  CholQR: the shift of Fukaya et
        // al. (2020), 11 (m w + w (w + 1)) u ||X||_F^2, in the first step.
        sh0 = op == OP_CQR1 ? 11.0 * ((double)a.m * wb + (double)wb * (wb + 1)) * u * t0
              : qr          ? 0.0
                            : a.pshift * u * t0;
        sh1 = a.pshift * u * t1;
    }
    for (int e = tid; e < W * W; e += nt) {
        const int i = e & (W - 1), j = e >> LW;
        double x = 0.0, y = 0.0, z = 0.0;
        if (i <= j && j < wb) x = P[bot + i + (int64_t)j * na];
        if (i < wb && j < wn) y = Pn[c + i + (int64_t)j * na];
        if (pyth && i <= j && j < wn) z = Pn[c + wb + i + (int64_t)j * na];
        M[i * L + j] = x + (i == j ? sh0 : 0.0);
        M[i * L + W + j] = y;
        M[(W + i) * L + W + j] = z + (i == j ? sh1 : 0.0);
    }
    // Minus the prefix Gram.
    if (!qr) {
        const GramPlan<W> gp(wb, wn, pyth);
        d_gram<W>(nt, gp, c, wb, wn, P, na, Z);
        __syncthreads();
        for (int e = tid; e < gp.np * 256; e += nt) {
            int p, q;
            gp.pair(e >> 8, &p, &q);
            const double *z = Z + 256 * ((e >> 8) * gp.KS) + (e & 255);
            double s = z[0];
            for (int k = 1; k < gp.KS; k++) s += z[256 * k];
            const int i = (p < gp.nY ? 16 * p : W + 16 * (p - gp.nY)) + ((e >> 4) & 15);
            const int j = (q < gp.nY ? 16 * q : W + 16 * (q - gp.nY)) + (e & 15);
            M[i * L + j] -= s;
        }
    }
    __syncthreads();
    // Wave 0: this block's factor with the lag correction
    // S_bot = Om^{-T} (..) beside it, and S_bot^T S_bot off the next block's
    // Gram; the others: the prefix rows of R.
    if (wave == 0) {
        wave_chol<W>(wb, wn > 0 ? W + wn : wb, M, rc, info);
        if (pyth) wave_syrk<W>(wb, W, wn, W, wn, true, M);
    } else if (!qr) {
        d_r_rows<W>(nt, 1, mode, c, wb, wn, P, na, a.Sig, Rb, a.ldR);
    }
    __syncthreads();
    const bool fold = a.Cout && wn > 0 && !(a.flags & F_SEQ);
    if (wave == 0 && pyth) {
        // The next block's factor.
        wave_chol<W>(wn, wn, M + W * L + W, rc + W, info + 1);
    } else if (wave == 1 && fold) {
        wave_solve_z2<W>(wb, wn, M, Z);
    } else if (wave >= 2) {
        const int t = tid - 128, n = nt - 128;
        d_write_slot<W>(t, n, wb, info[0] > 0 ? info[0] - 1 : wb, M, rc, qr ? a.Cq + (op - OP_CQR1) * kSlot : close ? a.Om : a.Sig);
        // R_bb = Omega Sigma (Omega in the A-1S form); S_bot to R and P.
        if (close) {
            if (mode == 2) d_trmm<W>(t, n, wb, M, L, a.Sig, Rb + c, 1, a.ldR);
            for (int e = t; e < W * W; e += n) {
                const int i = e & (W - 1), j = e >> LW;
                if (mode == 1 && i < wb && j < wb) Rb[c + i + (int64_t)j * a.ldR] = M[i * L + j];
                if (i < wb && j < wn) {
                    const double v = M[i * L + W + j];
                    Pn[c + i + (int64_t)j * na] = v;
                    Rb[c + i + (int64_t)(wb + j) * a.ldR] = v;
                }
            }
        }
        if (op == OP_CQR3) d_trmm<W>(t, n, wb, M, L, a.Cq + kSlot, Z, LZ, 1);
    }
    if (tid == 0) note_info(a.status, a.blk, info[0]);
    if (op == OP_CQR3) {
        // R3 R2 R1, and R_bb = (R3 R2 R1) Sigma (SRC/orth.c:537-541).
        double *RR = Z + W * LZ;
        __syncthreads();
        d_trmm<W>(tid, nt, wb, Z, LZ, a.Cq, RR, LZ, 1);
        __syncthreads();
        for (int e = tid; e < W * W; e += nt) {
            const int i = e & (W - 1), j = e >> LW;
            if (i < wb && j < wb) a.Rdst[i + (int64_t)j * a.ldRdst] = RR[i * LZ + j];
        }
        if (a.flags & F_RBB) d_trmm<W>(tid, nt, wb, RR, LZ, a.Sig, Rb + c, 1, a.ldR);
    }
    if (qr) return;
    if (pyth || fold) __syncthreads();
    if (pyth) {
        if (tid == 0) note_info(a.status, a.blk + 1, info[1]);
        d_write_slot<W>(tid, nt, wn, info[1] > 0 ? info[1] - 1 : wn, M + W * L + W, rc + W, a.Sig);
    }
    if (a.Cout) {
        // Next pass: the first group finalizes block b with [Y; 0] (closing
        // steps) or applies S (opening ones); the second is the first pass
        // of block b+1 with the prefix [Q Q^_b] and [S_top - Y Z2; Z2], which
        // equals Q S_top + Q_b S_bot without waiting for Q_b, or, in the
        // sequential form, S on the finished Q_b.
        const int k1 = op == OP_CLOSE_OPEN ? c + wb : c;
        d_emit<W>(nt, a.Cout, a.n1, a.S, k1, c, wb, wn, P, na, fold ? Z : M + W, fold ? LZ : L,
                  fold);
    }
}

}  // namespace orth
