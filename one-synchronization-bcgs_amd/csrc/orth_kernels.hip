// Device kernels of liborth_hip.so (gfx950) besides the fused passes
// (orth_pass*.hip, orth_mixed.hip) and the synchronization (orth_sync.hip).
//
//  k_update  row-local block updates, one row per lane, coefficients read as
//            wave-uniform (scalar) loads
//  k_upd     the schedules' paired block updates on v_mfma_f64_16x16x4f64
//            (shared prefix reads, blocked MFMA triangular solve)
//  k_proj    A^T B over a row slab on v_mfma_f64_16x16x4f64, 16-row tiles
//            staged through LDS with the next tile prefetched into
//            registers; one partial per workgroup
//  k_resid   ||Q R - X||_F and ||X||_F partial sums (accuracy harness)
#include "orth_kernels.h"

#include <math.h>
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "orth_device.h"

namespace orth {

// ---------------------------------------------------------------------------
// Row-local updates
// ---------------------------------------------------------------------------

template <int S>
__device__ __forceinline__ void apply_upd(double *__restrict__ xr, int64_t ldX,
                                          const Upd &u)
{
    double acc[S];
#pragma unroll
    for (int i = 0; i < S; i++) acc[i] = (i < u.w) ? xr[(u.col0 + i) * ldX] : 0.0;
    const int c = u.c;
    int j = 0;
    for (; j + 4 <= c; j += 4) {
        const double q0 = xr[(int64_t)j * ldX];
        const double q1 = xr[(int64_t)(j + 1) * ldX];
        const double q2 = xr[(int64_t)(j + 2) * ldX];
        const double q3 = xr[(int64_t)(j + 3) * ldX];
        const double *w = u.W + j;
#pragma unroll
        for (int i = 0; i < S; i++) {
            const double *wi = w + i * u.ldW;
            double a = acc[i];
            a = fma(-q0, wi[0], a);
            a = fma(-q1, wi[1], a);
            a = fma(-q2, wi[2], a);
            a = fma(-q3, wi[3], a);
            acc[i] = a;
        }
    }
    for (; j < c; j++) {
        const double q = xr[(int64_t)j * ldX];
#pragma unroll
        for (int i = 0; i < S; i++) acc[i] = fma(-q, u.W[j + i * u.ldW], acc[i]);
    }
    if (u.T) {
        // Row-wise forward substitution with the upper factor (dtrsm R,U,N,N).
#pragma unroll
        for (int i = 0; i < S; i++) {
            if (i < u.w) {
                double v = acc[i];
#pragma unroll
                for (int l = 0; l < i; l++) v = fma(-acc[l], u.T[l + i * kLdT], v);
                acc[i] = v * (1.0 / u.T[i + i * kLdT]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < S; i++)
        if (i < u.w) xr[(u.col0 + i) * ldX] = acc[i];
}

template <int S>
__global__ __launch_bounds__(256) void k_update(double *X, int64_t ldX, int64_t m,
                                                Upd u0, Upd u1, int nupd)
{
    const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (r >= m) return;
    double *xr = X + r;
    apply_upd<S>(xr, ldX, u0);
    if (nupd > 1) apply_upd<S>(xr, ldX, u1);
}

// Block updates on FP64 MFMA (s = 16, 32: NT = s / 16 column tiles).  Each
// wave owns 16 MT rows.  The products over the shared prefix [0, u0.c) of
// both updates run in one K-loop (one read of the prefix); the triangular
// solve X <- X T^{-1} is the blocked scheme of the s = 16 pass (one MFMA per
// 4-column block with the row blocks [D_b | -D_b T(b, >)] the Cholesky step
// stores beside T).  u1's prefix is u0's prefix followed by u0's block
// (checked by the host): that block's final values go from registers
// through LDS into u1's product.  No workgroup barrier: waves past the last
// row return.
// TWO: u1 follows u0 (the pairing); else u0 alone.
template <int NT, int MT, bool TWO>
__global__ __launch_bounds__(256) void k_upd(double *X, int64_t ldX, int64_t m, Upd u0, Upd u1)
{
    constexpr int S = 16 * NT, LDY = S + 1, RW = 16 * MT;
    __shared__ double ys_all[4][RW * LDY];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int64_t row0 = ((int64_t)blockIdx.x * 4 + wave) * RW;
    if (row0 >= m) return;
    double *ys = ys_all[wave];
    int64_t ra[MT];  // A-operand row of this lane per M-tile (clamped to the slab)
#pragma unroll
    for (int t = 0; t < MT; t++) ra[t] = min(row0 + 16 * t + li, m - 1);
    dbl4 z0[MT][NT], z1[TWO ? MT : 1][NT];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int n = 0; n < NT; n++) {
            z0[t][n] = dbl4{0.0, 0.0, 0.0, 0.0};
            if constexpr (TWO) z1[t][n] = dbl4{0.0, 0.0, 0.0, 0.0};
        }
    // Z += X(:, j0:j0+4) W(j0:j0+4, :) for j0 in [lo, hi), for u0 and (when
    // paired) u1: A lane (li, lk) holds X(row li, j0 + lk), B lane holds
    // W(j0 + lk, 16 n + li); columns past hi read column hi - 1 with zero
    // coefficients.
    auto kloop = [&](int lo, int hi) {
#pragma unroll 4
        for (int j0 = lo; j0 < hi; j0 += 4) {
            const int j = j0 + lk;
            const bool jok = j < hi;
            const int64_t jc = jok ? j : hi - 1;
            double a[MT];
#pragma unroll
            for (int t = 0; t < MT; t++) a[t] = X[ra[t] + jc * ldX];
#pragma unroll
            for (int n = 0; n < NT; n++) {
                const int col = 16 * n + li;
                {
                    const double b = jok && col < u0.w ? u0.W[j + (int64_t)col * u0.ldW] : 0.0;
#pragma unroll
                    for (int t = 0; t < MT; t++)
                        z0[t][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], b, z0[t][n], 0, 0, 0);
                }
                if constexpr (TWO) {
                    const double b = jok && col < u1.w ? u1.W[j + (int64_t)col * u1.ldW] : 0.0;
#pragma unroll
                    for (int t = 0; t < MT; t++)
                        z1[t][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], b, z1[t][n], 0, 0, 0);
                }
            }
        }
    };
    // Y = X(:, col0:col0+w) - Z, then Y <- Y T^{-1}, then store (D layout:
    // lane (li, lk) value v is row lk + 4 v, column 16 n + li).
    auto finish = [&](const Upd &u, auto &z) {
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int n = 0; n < NT; n++) {
                const int col = 16 * n + li;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int64_t row = row0 + 16 * t + lk + 4 * v;
                    const double x = row < m && col < u.w ? X[row + (u.col0 + col) * ldX] : 0.0;
                    z[t][n][v] = x - z[t][n][v];
                }
            }
        if (u.T) {
            const double *T = u.T;
            for (int b = 0; b < (u.w + 3) >> 2; b++) {
                const int nt = b >> 2, cb = b & 3;
                // Block b's current values go through LDS to become A operands.
                if ((li >> 2) == cb) {
#pragma unroll
                    for (int t = 0; t < MT; t++)
#pragma unroll
                        for (int n = 0; n < NT; n++)
                            if (n == nt) {
#pragma unroll
                                for (int v = 0; v < 4; v++)
                                    ys[(16 * t + lk + 4 * v) * LDY + 4 * b + (li & 3)] = z[t][n][v];
                            }
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                double av[MT];
#pragma unroll
                for (int t = 0; t < MT; t++) av[t] = ys[(16 * t + li) * LDY + 4 * b + lk];
#pragma unroll
                for (int n = 0; n < NT; n++) {
                    if (n < nt) continue;
                    const double bv = T[kSlotW + 128 * b + lk * kLdT + 16 * n + li];
#pragma unroll
                    for (int t = 0; t < MT; t++) {
                        if (n == nt && (li >> 2) == cb) z[t][n] = dbl4{0.0, 0.0, 0.0, 0.0};
                        z[t][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[t], bv, z[t][n], 0, 0, 0);
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
        }
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int n = 0; n < NT; n++) {
                const int col = 16 * n + li;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int64_t row = row0 + 16 * t + lk + 4 * v;
                    if (row < m && col < u.w) X[row + (u.col0 + col) * ldX] = z[t][n][v];
                }
            }
    };
    if (u0.c > 0) kloop(0, u0.c);
    finish(u0, z0);
    if constexpr (TWO) {
        // u1 += (u0's finished block) W1(u0.c : u0.c + u0.w, :).
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int n = 0; n < NT; n++)
                if (16 * n + li < u0.w) {
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        ys[(16 * t + lk + 4 * v) * LDY + 16 * n + li] = z0[t][n][v];
                }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        for (int j0 = 0; j0 < u0.w; j0 += 4) {
            const int j = j0 + lk;
            const bool jok = j < u0.w;
            double av[MT];
#pragma unroll
            for (int t = 0; t < MT; t++) av[t] = jok ? ys[(16 * t + li) * LDY + j] : 0.0;
#pragma unroll
            for (int n = 0; n < NT; n++) {
                const int col = 16 * n + li;
                const double b = jok && col < u1.w ? u1.W[u0.c + j + (int64_t)col * u1.ldW] : 0.0;
#pragma unroll
                for (int t = 0; t < MT; t++)
                    z1[t][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[t], b, z1[t][n], 0, 0, 0);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        finish(u1, z1);
    }
}

// Paired updates, 32 rows per wave.
template <int NT>
hipError_t launch_upd_pair(double *X, int64_t ldX, int64_t m, const Upd *u, hipStream_t st)
{
    const int64_t rows = 4 * 16 * 2;
    k_upd<NT, 2, true><<<dim3((unsigned)((m + rows - 1) / rows)), dim3(256), 0, st>>>(X, ldX, m,
                                                                                    u[0], u[1]);
    return hipGetLastError();
}

hipError_t launch_update(int S, double *X, int64_t ldX, int64_t m,
                         const Upd *u, int nupd, hipStream_t st)
{
    if (m <= 0 || nupd <= 0) return hipSuccess;
    // The MFMA form takes the schedules' pairing (u1's prefix is u0's prefix
    // followed by u0's block), where it shares the prefix and coefficient
    // loads between the two products; single updates stay row-wise (there,
    // even at 64 rows per wave, the MFMA form's coefficient loads cost more
    // than it saves).
    const bool paired = nupd == 2 && u[0].col0 == u[0].c && u[1].c == u[0].c + u[0].w;
    if ((S == 16 || S == 32) && paired && !getenv("ORTH_UPDATE_ROWWISE"))
        return S == 16 ? launch_upd_pair<1>(X, ldX, m, u, st) : launch_upd_pair<2>(X, ldX, m, u, st);
    dim3 grid((unsigned)((m + 255) / 256)), block(256);
    Upd u1 = nupd > 1 ? u[1] : u[0];
    switch (S) {
    case 4: k_update<4><<<grid, block, 0, st>>>(X, ldX, m, u[0], u1, nupd); break;
    case 8: k_update<8><<<grid, block, 0, st>>>(X, ldX, m, u[0], u1, nupd); break;
    case 16: k_update<16><<<grid, block, 0, st>>>(X, ldX, m, u[0], u1, nupd); break;
    case 32: k_update<32><<<grid, block, 0, st>>>(X, ldX, m, u[0], u1, nupd); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Projection A^T B on FP64 MFMA
// ---------------------------------------------------------------------------

constexpr int kRT = 16;       // rows per LDS tile
constexpr int kLdsLd = kRT + 1;  // padded column stride in LDS (doubles)
constexpr int kMaxTilesPerWave = 12;
constexpr int kMaxLdsCols = 20 * 16;

ProjPlan plan_proj(int64_t m, int64_t na, int64_t nb, int target_wg)
{
    ProjPlan p;
    p.Ma = (int)((na + 15) / 16);
    p.Nb = (int)((nb + 15) / 16);
    p.gb = p.Nb <= 4 ? p.Nb : (p.Nb < 8 ? p.Nb : 8);
    int ga = 4 * kMaxTilesPerWave / p.gb;
    if (ga > kMaxLdsCols / 16 - p.gb) ga = kMaxLdsCols / 16 - p.gb;
    if (ga > p.Ma) ga = p.Ma;
    if (ga < 1) ga = 1;
    p.ga = ga;
    p.ngy = ((p.Ma + p.ga - 1) / p.ga) * ((p.Nb + p.gb - 1) / p.gb);
    int64_t chunks = (m + kRT - 1) / kRT;
    int64_t want = target_wg / p.ngy;
    if (want < 1) want = 1;
    if (want > chunks) want = chunks;
    if (want < 1) want = 1;
    int64_t rows = (m + want - 1) / want;
    rows = ((rows + kRT - 1) / kRT) * kRT;
    if (rows < kRT) rows = kRT;
    p.rows_per = rows;
    p.nwg = (int)((m + rows - 1) / rows);
    if (p.nwg < 1) p.nwg = 1;
    p.lds_bytes = (size_t)(p.ga + p.gb) * 16 * kLdsLd * sizeof(double);
    return p;
}

// PF: load steps per tile (16 columns each), at least the column group's
// width / 16; every step loads (columns past the group read column a0).
template <int PF>
__global__ __launch_bounds__(256) void k_proj(const double *__restrict__ X, int64_t ldX,
                                              int64_t m, int64_t a0, int na, int64_t b0,
                                              int nb, int Ma, int Nb, int ga, int gb,
                                              int64_t rows_per, double *__restrict__ part)
{
    extern __shared__ double lds[];
    const int ngb = (Nb + gb - 1) / gb;
    const int gy = blockIdx.y;
    const int ta0 = (gy / ngb) * ga, tb0 = (gy % ngb) * gb;
    const int nta = min(ga, Ma - ta0), ntb = min(gb, Nb - tb0);
    const int colsA = nta * 16, ncol = colsA + ntb * 16;
    const int ntiles = nta * ntb;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int li = lane & 15, lk = lane >> 4;

    dbl4 acc[kMaxTilesPerWave];
#pragma unroll
    for (int t = 0; t < kMaxTilesPerWave; t++) acc[t] = dbl4{0.0, 0.0, 0.0, 0.0};

    const int64_t rb = (int64_t)blockIdx.x * rows_per;
    const int64_t re = min(m, rb + rows_per);
    // The next tile is prefetched into registers while the current one is
    // multiplied.  Element tid + 256 i of a tile is column (tid >> 4) + 16 i,
    // row tid & 15, so load step i of wave w moves columns 4 w + 16 i .. + 3,
    // which never straddle the A / B boundary (colsA is a multiple of 16):
    // the step's first column is wave-uniform and each lane adds its column
    // offset (lane >> 4).  Every lane loads unconditionally from a valid
    // address (columns past na / nb read column a0, rows past the end the
    // last row); the LDS store zeroes those elements.
    const int rr = threadIdx.x & (kRT - 1), lc = lane >> 4;
    const int64_t lcoff = (int64_t)lc * ldX;
    double pf[PF];
    // Group column cl (wave-uniform cw = cl - lc) -> matrix column and validity.
    auto colbase = [&](int cw, int64_t &base, bool &lok) {
        if (cw < colsA) {
            const int ac = ta0 * 16 + cw;
            lok = ac + lc < na;
            base = ac < na ? a0 + ac : a0;
        } else {
            const int bc = tb0 * 16 + (cw - colsA);
            lok = bc + lc < nb;
            base = bc < nb ? b0 + bc : a0;
        }
    };
    auto load = [&](int64_t r0) {
        int64_t rowc = min(r0 + rr, re - 1);
        // Opaque to the optimizer, so the addresses are not hoisted.
        asm volatile("" : "+v"(rowc));
#pragma unroll
        for (int i = 0; i < PF; i++) {
            const int cw = 4 * wave + 16 * i;
            int64_t base = a0;
            bool lok = false;
            if (cw < ncol) colbase(cw, base, lok);
            pf[i] = X[base * ldX + (lok ? lcoff : 0) + rowc];
        }
    };
    if (rb < re) load(rb);
    for (int64_t r0 = rb; r0 < re; r0 += kRT) {
        __syncthreads();
        const bool rok = r0 + rr < re;
#pragma unroll
        for (int i = 0; i < PF; i++) {
            const int cw = 4 * wave + 16 * i;
            if (cw < ncol) {
                int64_t base;
                bool lok;
                colbase(cw, base, lok);
                lds[(cw + lc) * kLdsLd + rr] = lok && rok ? pf[i] : 0.0;
            }
        }
        __syncthreads();
        if (r0 + kRT < re) load(r0 + kRT);
#pragma unroll
        for (int ks = 0; ks < kRT / 4; ks++) {
            const int rk = ks * 4 + lk;
#pragma unroll
            for (int t = 0; t < kMaxTilesPerWave; t++) {
                const int tile = wave + 4 * t;
                if (tile < ntiles) {
                    const int ta = tile / ntb, tb = tile - ta * ntb;
                    const double a = lds[(ta * 16 + li) * kLdsLd + rk];
                    const double b = lds[(colsA + tb * 16 + li) * kLdsLd + rk];
                    acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc[t], 0, 0, 0);
                }
            }
        }
    }
    // D layout of v_mfma_f64_16x16x4f64: lane (li, lk), value v holds row
    // lk + 4 v, column li of the tile.
    double *out = part + (int64_t)blockIdx.x * na * nb;
#pragma unroll
    for (int t = 0; t < kMaxTilesPerWave; t++) {
        const int tile = wave + 4 * t;
        if (tile < ntiles) {
            const int ta = tile / ntb, tb = tile - ta * ntb;
            const int j = (tb0 + tb) * 16 + li;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = (ta0 + ta) * 16 + lk + 4 * v;
                if (i < na && j < nb) out[i + (int64_t)j * na] = acc[t][v];
            }
        }
    }
}

hipError_t launch_proj(const ProjPlan &pl, const double *X, int64_t ldX, int64_t m,
                       int64_t a0, int64_t na, int64_t b0, int64_t nb, double *part,
                       hipStream_t st)
{
    dim3 grid(pl.nwg, pl.ngy), block(256);
    const int steps = (pl.ga + pl.gb + 3) / 4 * 4;  // 16-column load steps, rounded up to 4
#define ORTH_PROJ(P)                                                                        \
    case P:                                                                                 \
        k_proj<P><<<grid, block, pl.lds_bytes, st>>>(X, ldX, m, a0, (int)na, b0, (int)nb,   \
                                                     pl.Ma, pl.Nb, pl.ga, pl.gb,            \
                                                     pl.rows_per, part);                    \
        break;
    switch (steps) {
        ORTH_PROJ(4) ORTH_PROJ(8) ORTH_PROJ(12) ORTH_PROJ(16) ORTH_PROJ(20)
    default: return hipErrorInvalidValue;
    }
#undef ORTH_PROJ
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Streaming probes (measurement of the device's streaming ceiling)
// ---------------------------------------------------------------------------

typedef double dbl2p __attribute__((ext_vector_type(2)));

// dst = src over n2 16-byte elements, 8 non-temporal loads in flight per
// thread before the stores.
__global__ __launch_bounds__(256) void k_probe_copy(const dbl2p *__restrict__ src,
                                                    dbl2p *__restrict__ dst, int64_t n2)
{
    constexpr int U = 8;
    const int64_t stride = (int64_t)gridDim.x * 256 * U;
    for (int64_t base = (int64_t)blockIdx.x * 256 * U + threadIdx.x; base < n2; base += stride) {
        dbl2p v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t i = base + (int64_t)u * 256;
            v[u] = i < n2 ? __builtin_nontemporal_load(src + i) : dbl2p{0.0, 0.0};
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t i = base + (int64_t)u * 256;
            if (i < n2) __builtin_nontemporal_store(v[u], dst + i);
        }
    }
}

// Reads n2 16-byte elements; one per-workgroup sum goes to part[blockIdx.x]
// (so that the loads are kept).
__global__ __launch_bounds__(256) void k_probe_read(const dbl2p *__restrict__ src, double *part,
                                                    int64_t n2)
{
    constexpr int U = 8;
    __shared__ double red[256];
    const int64_t stride = (int64_t)gridDim.x * 256 * U;
    double t = 0.0;
    for (int64_t base = (int64_t)blockIdx.x * 256 * U + threadIdx.x; base < n2; base += stride) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t i = base + (int64_t)u * 256;
            if (i < n2) {
                const dbl2p v = __builtin_nontemporal_load(src + i);
                t += v.x + v.y;
            }
        }
    }
    red[threadIdx.x] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int k = 0; k < 256; k++) s += red[k];
        part[blockIdx.x] = s;
    }
}

hipError_t launch_stream_probe(int mode, double *dst, const double *src, int64_t bytes,
                               double *part, int nwg, hipStream_t st)
{
    const int64_t n2 = bytes / 16;
    if (n2 < 1 || nwg < 1) return hipErrorInvalidValue;
    if (mode == 0)
        k_probe_copy<<<dim3(nwg), dim3(256), 0, st>>>((const dbl2p *)src, (dbl2p *)dst, n2);
    else
        k_probe_read<<<dim3(nwg), dim3(256), 0, st>>>((const dbl2p *)src, part, n2);
    return hipGetLastError();
}

// Q (m x n, ld ldq) = X32 widened exactly to FP64.
__global__ __launch_bounds__(256) void k_widen(const float *__restrict__ x, int64_t ldx,
                                                double *__restrict__ q, int64_t ldq, int64_t m,
                                                int64_t n)
{
    const int64_t total = m * n;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = e % m, j = e / m;
        q[i + j * ldq] = (double)x[i + j * ldx];
    }
}

hipError_t launch_widen(const float *x, int64_t ldx, double *q, int64_t ldq, int64_t m, int64_t n,
                        hipStream_t st)
{
    const int64_t total = m * n;
    const int nb = (int)std::min<int64_t>((total + 255) / 256, 8192);
    k_widen<<<dim3(std::max(nb, 1)), dim3(256), 0, st>>>(x, ldx, q, ldq, m, n);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_fill(double *p, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        p[i] = 0.0;
}

hipError_t launch_fill(double *p, size_t n, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    size_t g = (n + 255) / 256;
    if (g > 4096) g = 4096;
    k_fill<<<dim3((unsigned)g), dim3(256), 0, st>>>(p, n);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Residual of the accuracy harness
// ---------------------------------------------------------------------------

constexpr int kResidWG = 1024;

int resid_wg_count(int64_t m)
{
    int64_t g = (m + 255) / 256;
    return (int)(g < kResidWG ? g : kResidWG);
}

__global__ __launch_bounds__(256) void k_resid(int64_t m, int n, const double *__restrict__ X,
                                               int64_t ldX, const double *__restrict__ Q,
                                               int64_t ldQ, const double *__restrict__ R,
                                               int64_t ldR, double *part2)
{
    __shared__ double red[2][256];
    double sr = 0.0, sx = 0.0;
    for (int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x; r < m;
         r += (int64_t)gridDim.x * 256) {
        for (int j0 = 0; j0 < n; j0 += 16) {
            double t[16];
#pragma unroll
            for (int jj = 0; jj < 16; jj++) {
                const int j = j0 + jj;
                const double x = j < n ? X[r + j * ldX] : 0.0;
                sx = fma(x, x, sx);
                t[jj] = -x;
            }
            for (int i = 0; i < n; i++) {
                const double q = Q[r + i * ldQ];
#pragma unroll
                for (int jj = 0; jj < 16; jj++) {
                    const int j = j0 + jj;
                    if (j < n) t[jj] = fma(q, R[i + j * ldR], t[jj]);
                }
            }
#pragma unroll
            for (int jj = 0; jj < 16; jj++) sr = fma(t[jj], t[jj], sr);
        }
    }
    red[0][threadIdx.x] = sr;
    red[1][threadIdx.x] = sx;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (threadIdx.x < h) {
            red[0][threadIdx.x] += red[0][threadIdx.x + h];
            red[1][threadIdx.x] += red[1][threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part2[2 * blockIdx.x] = red[0][0];
        part2[2 * blockIdx.x + 1] = red[1][0];
    }
}

hipError_t launch_resid(int64_t m, int64_t n, const double *X, int64_t ldX, const double *Q,
                        int64_t ldQ, const double *R, int64_t ldR, double *part2,
                        hipStream_t st)
{
    k_resid<<<dim3(resid_wg_count(m)), dim3(256), 0, st>>>(m, (int)n, X, ldX, Q, ldQ, R, ldR,
                                                           part2);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Accuracy harness: the Gram Q^T Q with compensated accumulation (Dot2 of
// Ogita, Rump and Oishi, "Accurate sum and dot product", SIAM J. Sci. Comput.
// 26 (2005): TwoProduct by FMA, TwoSum, the error terms summed in FP64), so
// that the Gram's own rounding stays far below the loss of orthogonality it
// measures.  Workgroup (x, y): row chunk x, 64 x 64 block y of the upper
// block triangle; thread t owns the 16 pairs (I0 + 4 (t % 16) + di,
// J0 + 4 (t / 16) + dj).  part: (hi, lo) of each pair, per chunk and block.
// ---------------------------------------------------------------------------
constexpr int kGramRows = 32;

__global__ __launch_bounds__(256) void k_gram_dd(const double *__restrict__ Q, int64_t ldQ,
                                                 int64_t m, int n, int64_t rows_per,
                                                 double *__restrict__ part)
{
#pragma clang fp contract(off)
    __shared__ double sa[kGramRows][65], sb[kGramRows][65];
    const int t = threadIdx.x;
    const int nb = (n + 63) / 64;
    // Block y -> (I, J), I <= J, row-major over the upper block triangle.
    int y = blockIdx.y, I = 0;
    while (y >= nb - I) {
        y -= nb - I;
        I++;
    }
    const int J = I + y, I0 = 64 * I, J0 = 64 * J;
    const int ti = 4 * (t % 16), tj = 4 * (t / 16);
    double hi[16], lo[16];
#pragma unroll
    for (int k = 0; k < 16; k++) hi[k] = lo[k] = 0.0;
    const int64_t rb = (int64_t)blockIdx.x * rows_per, re = min(m, rb + rows_per);
    for (int64_t r0 = rb; r0 < re; r0 += kGramRows) {
        for (int e = t; e < kGramRows * 64; e += 256) {
            const int c = e / kGramRows, r = e % kGramRows;
            const bool in = r0 + r < re;
            sa[r][c] = in && I0 + c < n ? Q[r0 + r + (int64_t)(I0 + c) * ldQ] : 0.0;
            sb[r][c] = in && J0 + c < n ? Q[r0 + r + (int64_t)(J0 + c) * ldQ] : 0.0;
        }
        __syncthreads();
        for (int r = 0; r < kGramRows; r++) {
            double a[4], b[4];
#pragma unroll
            for (int d = 0; d < 4; d++) {
                a[d] = sa[r][ti + d];
                b[d] = sb[r][tj + d];
            }
#pragma unroll
            for (int di = 0; di < 4; di++)
#pragma unroll
                for (int dj = 0; dj < 4; dj++) {
                    const int k = 4 * di + dj;
                    const double p = a[di] * b[dj];
                    const double pe = __builtin_fma(a[di], b[dj], -p);
                    const double sum = hi[k] + p;
                    const double bp = sum - hi[k];
                    const double se = (hi[k] - (sum - bp)) + (p - bp);
                    hi[k] = sum;
                    lo[k] += se + pe;
                }
        }
        __syncthreads();
    }
    double *o = part + ((int64_t)(blockIdx.x * gridDim.y + blockIdx.y) * 256 + t) * 32;
#pragma unroll
    for (int k = 0; k < 16; k++) {
        o[2 * k] = hi[k];
        o[2 * k + 1] = lo[k];
    }
}

int gram_dd_chunks(int64_t m)
{
    return (int)std::max<int64_t>(1, std::min<int64_t>(64, (m + 4095) / 4096));
}

hipError_t launch_gram_dd(const double *Q, int64_t ldQ, int64_t m, int64_t n, double *part,
                          hipStream_t st)
{
    const int nch = gram_dd_chunks(m), nb = (int)((n + 63) / 64);
    int64_t rows = (m + nch - 1) / nch;
    rows = (rows + kGramRows - 1) / kGramRows * kGramRows;
    k_gram_dd<<<dim3(nch, nb * (nb + 1) / 2), dim3(256), 0, st>>>(Q, ldQ, m, (int)n, rows, part);
    return hipGetLastError();
}

}  // namespace orth
