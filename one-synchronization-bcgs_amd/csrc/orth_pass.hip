// The 256-thread fused passes (gfx950): the generic pass for any block width
// and the s = 16 form with compile-time tile counts.
#include "orth_kernels.h"

#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "orth_device.h"
#include "orth_tail.h"

namespace orth {

// ---------------------------------------------------------------------------
// Fused pass: updates + projection in one sweep over the row slab
// ---------------------------------------------------------------------------

constexpr int kPT = kPassRows;                   // rows per tile (32)
constexpr int kPLd = kPT + 1;                    // padded column stride (doubles)
constexpr int kPF = kPassMaxCols * kPT / 256;    // prefetch registers per thread
constexpr int kPassMaxTiles = 12;                // projection tiles per wave
constexpr int kPassMaxC = 8192;                  // doubles of C held in LDS

size_t pass_lds_bytes(const PassArgs &a, int F)
{
    if (a.ncols > kPassMaxCols || a.wl < a.ncols || a.wl > kPassMaxCols + 32) return 0;
    const int k1p = (a.k1 + 3) & ~3;
    if ((size_t)k1p * a.n1 > (size_t)kPassMaxC || k1p > a.wl) return 0;
    if (a.k1 > 0 && (a.n1 % 16 != 0 || (F * kPT / 16) * (a.n1 / 16) > 8)) return 0;
    if (a.na > 0) {
        const int Ma = (a.na + 15) / 16, Nb = (a.nb + 15) / 16;
        if (Ma * Nb > 4 * kPassMaxTiles) return 0;
        if (a.a0 + Ma * 16 > a.wl || a.b0 + Nb * 16 > a.wl) return 0;
    }
    for (int g = 0; g < a.ngrp; g++)
        if (a.g[g].w > kMaxS || a.g[g].t0 + a.g[g].w > a.ncols) return 0;
    return ((size_t)a.wl * (F * kPT + 1) + (size_t)k1p * a.n1 + 2 * kMaxS * kMaxS) * sizeof(double);
}

// Waves per SIMD (= 256-thread workgroups per CU) the generic pass is
// compiled for: the wide instance uses up to 512 registers per lane (one
// workgroup per CU); the narrow one fits three (S <= 8) or two (S = 16).
constexpr int pass_waves(int S, int MT) { return MT > 4 || S > 16 ? 1 : S <= 8 ? 3 : 2; }

// MT: projection tiles per wave, PF: prefetch registers per thread.  The
// narrow instance (fewer of both) fits several workgroups per CU.  V2: every
// lane moves two consecutive rows with one 16-byte load (even ldX and m,
// 16-byte aligned slab).  F: rows per tile = 32 F (the narrow instance with
// few columns takes longer runs of each column per tile).
template <int S, int MT = kPassMaxTiles, int PF = kPF, bool V2 = false, int F = 1>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(
    pass_waves(S, MT), pass_waves(S, MT)))) void k_pass(PassArgs a)
{
    constexpr int TS = kPT * F, PLD = TS + 1;
    extern __shared__ double sm[];
    const uint64_t kst = kernarg_stash();
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int li = lane & 15, lk = lane >> 4;
    const int k1p = (a.k1 + 3) & ~3;
    double *tile = sm;
    double *Cs = tile + a.wl * PLD;
    double *Ts = Cs + k1p * a.n1;  // one S x S factor per group, ld S

    for (int e = tid; e < k1p * a.n1; e += 256) Cs[e] = a.C[e];
    for (int g = 0; g < a.ngrp; g++) {
        const double *T = a.g[g].T;
        const int w = a.g[g].w;
        if (T)
            for (int e = tid; e < S * S; e += 256) {
                const int i = e % S, j = e / S;
                Ts[g * S * S + e] = (i < w && j < w) ? T[i + j * kLdT] : 0.0;
            }
    }
    for (int e = tid; e < (a.wl - a.ncols) * TS; e += 256)
        tile[(a.ncols + e / TS) * PLD + (e % TS)] = 0.0;

    const int Ma = (a.na + 15) >> 4, Nb = (a.nb + 15) >> 4;
    const int ntiles = a.na > 0 ? Ma * Nb : 0;

    dbl4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) acc[t] = dbl4{0.0, 0.0, 0.0, 0.0};

    const int64_t rb = (int64_t)blockIdx.x * a.rows_per;
    const int64_t re = min(a.m, rb + a.rows_per);
    // Load step i moves columns lcol + CPS i: LPC = TS / VR lanes per column,
    // VR consecutive rows per lane, so each group of LPC lanes reads TS
    // consecutive rows of one column.  A wave's lanes touch at most four
    // consecutive columns; the loads are addressed from a wave-uniform base
    // (the wave's first column) plus one 32-bit byte offset per lane (below
    // 8 (3 ldX + TS) bytes; the host keeps ldX under 2^27), so no per-step
    // 64-bit lane address is kept.  Every lane loads unconditionally (one
    // code path, so no register copies or zero defaults wait for loads or
    // stores in flight): lanes past the last row re-read the last valid
    // row(s), and the LDS store zeroes them.  With V2 the row count of every
    // tile is even.
    typedef double dbl2v __attribute__((ext_vector_type(2)));
    using PV = typename std::conditional<V2, dbl2v, double>::type;
    constexpr int VR = V2 ? 2 : 1, NPF = PF / VR;
    constexpr int LPC = TS / VR, CPS = 256 / LPC;
    static_assert(LPC >= 16 && LPC <= 256 && 256 % LPC == 0, "lane mapping");
    PV pf[NPF];
    const int lrow = VR * (tid % LPC), lcol = tid / LPC;
    const int wcol = __builtin_amdgcn_readfirstlane(lcol);
    const uint32_t lb = 8u * (uint32_t)((lcol - wcol) * a.ldX + lrow);
    const int64_t wcolb = (int64_t)wcol * a.ldX * 8, cstep = (int64_t)CPS * a.ldX * 8;
    auto load = [&](int64_t r0) {
        const int rem = (int)min(re - r0, (int64_t)TS);
        // Opaque to the optimizer, so the addresses are not hoisted.
        uint32_t o = lb - 8u * (uint32_t)max(0, lrow - (rem - VR));
        asm volatile("" : "+v"(o));
        const char *b = (const char *)(a.X + r0) + wcolb;
#pragma unroll
        for (int i = 0; i < NPF; i++)
            if (lcol + CPS * i < a.ncols) pf[i] = *(const PV *)(b + i * cstep + o);
    };
    if (rb < re) load(rb);
    __syncthreads();

    for (int64_t r0 = rb; r0 < re; r0 += TS) {
        __syncthreads();
        const bool rok = lrow < min(re - r0, (int64_t)TS);
#pragma unroll
        for (int i = 0; i < NPF; i++)
            if (lcol + CPS * i < a.ncols) {
                double *d = tile + (lcol + CPS * i) * PLD + lrow;
                if constexpr (V2) {
                    d[0] = rok ? pf[i].x : 0.0;
                    d[1] = rok ? pf[i].y : 0.0;
                } else {
                    d[0] = rok ? pf[i] : 0.0;
                }
            }
        __syncthreads();
        if (r0 + TS < re) load(r0 + TS);

        if (a.ngrp > 0) {
            // Step 1 in one phase (all groups from the same product) or, in
            // sequential mode, one phase per group.
            const int nphase = a.seq ? a.ngrp : 1;
            for (int p = 0; p < nphase; p++) {
                const int glo = a.seq ? p : 0, ghi = a.seq ? p + 1 : a.ngrp;
                int zlo = 1 << 30, zhi = 0;
                for (int g = glo; g < ghi; g++) {
                    zlo = min(zlo, a.g[g].zoff);
                    zhi = max(zhi, a.g[g].zoff + a.g[g].w);
                }
                const int ntlo = zlo >> 4, nN = ((zhi + 15) >> 4) - ntlo;
                const int kp = a.seq ? ((a.g[p].k + 3) & ~3) : k1p;
                const int ncombo = a.k1 > 0 ? (TS / 16) * nN : 0;
                // Z = tile(:, 0:kp) C(:, N-tiles), one 16 x 16 tile of Z per combo.
                dbl4 z[2];
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    z[q] = dbl4{0.0, 0.0, 0.0, 0.0};
                    const int combo = wave + 4 * q;
                    if (combo < ncombo) {
                        const int mt = combo / nN, nt = ntlo + combo % nN;
                        const double *ap = tile + lk * PLD + mt * 16 + li;
                        const double *bp = Cs + lk * a.n1 + nt * 16 + li;
                        for (int ks = 0; ks < kp / 4; ks++)
                            z[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                ap[4 * ks * PLD], bp[4 * ks * a.n1], z[q], 0, 0, 0);
                    }
                }
                __syncthreads();
                // Subtract Z from the target blocks (D layout: row lk + 4v, col li).
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const int combo = wave + 4 * q;
                    if (combo < ncombo) {
                        const int mt = combo / nN, nt = ntlo + combo % nN;
                        const int zc = nt * 16 + li;
                        for (int g = glo; g < ghi; g++) {
                            const int off = zc - a.g[g].zoff;
                            if (off >= 0 && off < a.g[g].w) {
                                double *col = tile + (a.g[g].t0 + off) * PLD + mt * 16 + lk;
#pragma unroll
                                for (int v = 0; v < 4; v++) col[4 * v] -= z[q][v];
                            }
                        }
                    }
                }
                __syncthreads();
                // Row-wise forward substitution with each group's factor
                // (dtrsm_('R','U','N','N') on the rows of the tile).
                for (int task = tid; task < (ghi - glo) * TS; task += 256) {
                    const int g = glo + task / TS, row = task % TS;
                    if (a.g[g].T) {
                        const int w = a.g[g].w;
                        double *col = tile + a.g[g].t0 * PLD + row;
                        const double *Tg = Ts + g * S * S;
                        double x[S];
#pragma unroll
                        for (int i = 0; i < S; i++) x[i] = i < w ? col[i * PLD] : 0.0;
#pragma unroll
                        for (int i = 0; i < S; i++) {
                            if (i < w) {
                                double v = x[i];
#pragma unroll
                                for (int l = 0; l < i; l++) v = fma(-x[l], Tg[l + i * S], v);
                                x[i] = v * (1.0 / Tg[i + i * S]);
                            }
                        }
#pragma unroll
                        for (int i = 0; i < S; i++)
                            if (i < w) col[i * PLD] = x[i];
                    }
                }
                __syncthreads();
            }
            // Write the finished target blocks back to X.
            for (int g = 0; g < a.ngrp; g++) {
                const int t0 = a.g[g].t0;
                for (int e = tid; e < a.g[g].w * TS; e += 256) {
                    const int cc = e / TS, rr = e - cc * TS;
                    const int64_t row = r0 + rr;
                    if (row < re) a.X[row + (int64_t)(t0 + cc) * a.ldX] = tile[(t0 + cc) * PLD + rr];
                }
            }
        }

        // Step 2: projection partials.
        if (ntiles > 0) {
#pragma unroll
            for (int ks = 0; ks < TS / 4; ks++) {
                const int rr = 4 * ks + lk;
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    const int tl = wave + 4 * t;
                    if (tl < ntiles) {
                        const int ta = tl / Nb, tb = tl - ta * Nb;
                        const double av = tile[(a.a0 + ta * 16 + li) * PLD + rr];
                        const double bv = tile[(a.b0 + tb * 16 + li) * PLD + rr];
                        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, acc[t], 0, 0, 0);
                    }
                }
            }
        }
    }

    if (ntiles > 0) {
        double *out = a.part + (int64_t)blockIdx.x * a.na * a.nb;
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const int tl = wave + 4 * t;
            if (tl < ntiles) {
                const int ta = tl / Nb, tb = tl - ta * Nb;
                const int j = tb * 16 + li;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int i = ta * 16 + lk + 4 * v;
                    if (i < a.na && j < a.nb) out[i + (int64_t)j * a.na] = acc[t][v];
                }
            }
        }
    }
    pass_tail(a, sm, kst, 256);
}

// Block width 16, the benchmark shape: compile-time tile counts, 32-bit
// LDS offsets, four independent MFMA chains in step 1.  Wave w computes
// Z tile (rows 16 (w & 1), cols 16 (w >> 1)) in step 1 and projection tiles
// [w MT, (w+1) MT) x [0, NB) in step 2.
template <int MT, int NB>
__global__ __launch_bounds__(256) void k_pass16(PassArgs a)
{
    constexpr int S = 16, N1 = 32, LD = kPLd;
    extern __shared__ double sm[];
    const uint64_t kst = kernarg_stash();
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int li = lane & 15, lk = lane >> 4;
    const int k1p = (a.k1 + 3) & ~3;
    const int C0 = a.wl * LD, T0 = C0 + k1p * N1;

    for (int e = tid; e < k1p * N1; e += 256) sm[C0 + e] = a.C[e];
    for (int g = 0; g < a.ngrp; g++) {
        const double *T = a.g[g].T;
        const int w = a.g[g].w;
        if (T)
            for (int e = tid; e < S * S; e += 256) {
                const int i = e % S, j = e / S;
                sm[T0 + g * S * S + e] = (i < w && j < w) ? T[i + j * kLdT] : 0.0;
            }
    }
    for (int e = tid; e < (a.wl - a.ncols) * kPT; e += 256)
        sm[(a.ncols + e / kPT) * LD + (e % kPT)] = 0.0;

    const int Ma = (a.na + 15) >> 4;
    const bool proj = a.na > 0;
    const int mt1 = wave & 1, nt1 = wave >> 1;
    const int aoff1 = lk * LD + mt1 * 16 + li;
    const int boff1 = C0 + lk * N1 + nt1 * 16 + li;
    int aoff2[MT], boff2[NB];
#pragma unroll
    for (int i = 0; i < MT; i++) aoff2[i] = (a.a0 + (wave * MT + i) * 16 + li) * LD + lk;
#pragma unroll
    for (int j = 0; j < NB; j++) boff2[j] = (a.b0 + j * 16 + li) * LD + lk;

    dbl4 acc[MT][NB];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};

    const int64_t rb = (int64_t)blockIdx.x * a.rows_per;
    const int64_t re = min(a.m, rb + a.rows_per);
    const int nload = a.ncols * kPT;
    const double *Xl = a.X + (tid & (kPT - 1));
    double pf[kPF];
    auto load = [&](int64_t r0) {
        const bool full = r0 + kPT <= re;
#pragma unroll
        for (int i = 0; i < kPF; i++) {
            const int e = tid + 256 * i;
            if (e < nload) {
                const int64_t off = r0 + (int64_t)(e >> 5) * a.ldX;
                pf[i] = (full || r0 + (e & 31) < re) ? Xl[off] : 0.0;
            }
        }
    };
    if (rb < re) load(rb);

    for (int64_t r0 = rb; r0 < re; r0 += kPT) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kPF; i++) {
            const int e = tid + 256 * i;
            if (e < nload) sm[(e >> 5) * LD + (e & 31)] = pf[i];
        }
        __syncthreads();
        if (r0 + kPT < re) load(r0 + kPT);

        if (a.ngrp > 0) {
            const int nphase = a.seq ? a.ngrp : 1;
            for (int p = 0; p < nphase; p++) {
                const int glo = a.seq ? p : 0, ghi = a.seq ? p + 1 : a.ngrp;
                const int kp = a.seq ? ((a.g[p].k + 3) & ~3) : k1p;
                const bool mine = a.k1 > 0 && (!a.seq || nt1 == (a.g[p].zoff >> 4));
                dbl4 z = dbl4{0.0, 0.0, 0.0, 0.0};
                if (mine) {
                    dbl4 z1 = z, z2 = z, z3 = z;
                    const int nks = kp >> 2;
                    int ks = 0;
                    for (; ks + 4 <= nks; ks += 4) {
                        const int ao = aoff1 + 4 * ks * LD, bo = boff1 + 4 * ks * N1;
                        const double x0 = sm[ao], x1 = sm[ao + 4 * LD], x2 = sm[ao + 8 * LD],
                                     x3 = sm[ao + 12 * LD];
                        const double c0 = sm[bo], c1 = sm[bo + 4 * N1], c2 = sm[bo + 8 * N1],
                                     c3 = sm[bo + 12 * N1];
                        z = __builtin_amdgcn_mfma_f64_16x16x4f64(x0, c0, z, 0, 0, 0);
                        z1 = __builtin_amdgcn_mfma_f64_16x16x4f64(x1, c1, z1, 0, 0, 0);
                        z2 = __builtin_amdgcn_mfma_f64_16x16x4f64(x2, c2, z2, 0, 0, 0);
                        z3 = __builtin_amdgcn_mfma_f64_16x16x4f64(x3, c3, z3, 0, 0, 0);
                    }
                    for (; ks < nks; ks++)
                        z = __builtin_amdgcn_mfma_f64_16x16x4f64(sm[aoff1 + 4 * ks * LD],
                                                                 sm[boff1 + 4 * ks * N1], z, 0,
                                                                 0, 0);
                    z = (z + z1) + (z2 + z3);
                }
                __syncthreads();
                if (mine) {
                    const int zc = nt1 * 16 + li;
                    for (int g = glo; g < ghi; g++) {
                        const int off = zc - a.g[g].zoff;
                        if (off >= 0 && off < a.g[g].w) {
                            const int o = (a.g[g].t0 + off) * LD + mt1 * 16 + lk;
#pragma unroll
                            for (int v = 0; v < 4; v++) sm[o + 4 * v] -= z[v];
                        }
                    }
                }
                __syncthreads();
                // Row-wise forward substitution (dtrsm_('R','U','N','N')).
                if (tid < (ghi - glo) * kPT) {
                    const int g = glo + tid / kPT, row = tid % kPT;
                    if (a.g[g].T) {
                        const int w = a.g[g].w;
                        const int o = a.g[g].t0 * LD + row;
                        const int tg = T0 + g * S * S;
                        double x[S];
#pragma unroll
                        for (int i = 0; i < S; i++) x[i] = i < w ? sm[o + i * LD] : 0.0;
#pragma unroll
                        for (int i = 0; i < S; i++) {
                            if (i < w) {
                                double v = x[i];
#pragma unroll
                                for (int l = 0; l < i; l++) v = fma(-x[l], sm[tg + l + i * S], v);
                                x[i] = v * (1.0 / sm[tg + i + i * S]);
                            }
                        }
#pragma unroll
                        for (int i = 0; i < S; i++)
                            if (i < w) sm[o + i * LD] = x[i];
                    }
                }
                __syncthreads();
            }
            for (int g = 0; g < a.ngrp; g++) {
                const int t0 = a.g[g].t0;
                for (int e = tid; e < a.g[g].w * kPT; e += 256) {
                    const int cc = e >> 5, rr = e & 31;
                    if (r0 + rr < re)
                        a.X[r0 + rr + (int64_t)(t0 + cc) * a.ldX] = sm[(t0 + cc) * LD + rr];
                }
            }
        }

        if (proj) {
#pragma unroll
            for (int ks = 0; ks < kPT / 4; ks++) {
                double bv[NB], av[MT];
#pragma unroll
                for (int j = 0; j < NB; j++) bv[j] = sm[boff2[j] + 4 * ks];
#pragma unroll
                for (int i = 0; i < MT; i++) av[i] = sm[aoff2[i] + 4 * ks];
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < NB; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i], bv[j], acc[i][j],
                                                                        0, 0, 0);
            }
        }
    }

    if (proj) {
        double *out = a.part + (int64_t)blockIdx.x * a.na * a.nb;
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const int ta = wave * MT + i;
            if (ta < Ma) {
#pragma unroll
                for (int j = 0; j < NB; j++) {
                    const int col = j * 16 + li;
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const int row = ta * 16 + lk + 4 * v;
                        if (row < a.na && col < a.nb) out[row + (int64_t)col * a.na] = acc[i][j][v];
                    }
                }
            }
        }
    }
    pass_tail(a, sm, kst, 256);
}

// Tiles per wave of the s = 16 kernel for a pass, or 0 when it does not apply.
static int pass16_mt(const PassArgs &a)
{
    if (a.n1 != 32) return 0;
    if (a.na == 0) return 1;
    const int Ma = (a.na + 15) / 16, Nb = (a.nb + 15) / 16;
    if (Nb > 2) return 0;
    const int mt = (Ma + 3) / 4;
    if (mt > 5 || a.a0 + 64 * mt > a.wl) return 0;
    return mt;
}

template <int MT, int NB>
hipError_t launch_pass16_t(const PassArgs &a, size_t lds, int nwg, hipStream_t st)
{
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void *)k_pass16<MT, NB>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)(160 * 1024));
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    k_pass16<MT, NB><<<dim3(nwg), dim3(256), lds, st>>>(a);
    return hipGetLastError();
}

hipError_t launch_pass16(const PassArgs &a, size_t lds, int nwg, hipStream_t st)
{
    const int mt = pass16_mt(a);
    const int nb = a.na > 0 ? (a.nb + 15) / 16 : 1;
#define ORTH_P16(M)                                                                  \
    case M:                                                                          \
        return nb == 2 ? launch_pass16_t<M, 2>(a, lds, nwg, st)                     \
                       : launch_pass16_t<M, 1>(a, lds, nwg, st);
    switch (mt) {
        ORTH_P16(1)
        ORTH_P16(2)
        ORTH_P16(3)
        ORTH_P16(4)
        ORTH_P16(5)
    default: return hipErrorInvalidValue;
    }
#undef ORTH_P16
}

// The narrow generic pass: at most kNarrowCols columns and 4 projection
// tiles per wave.
constexpr int kNarrowCols = 160;
constexpr int kNarrowPF = kNarrowCols * kPT / 256;

bool pass_narrow(const PassArgs &a)
{
    const int Ma = (a.na + 15) / 16, Nb = (a.nb + 15) / 16;
    return a.ncols <= kNarrowCols && (a.na == 0 || Ma * Nb <= 4 * 4);
}

template <int S, int MT, int PF, bool V2 = false, int F = 1>
hipError_t launch_pass_v(const PassArgs &a, size_t lds, int nwg, hipStream_t st)
{
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void *)k_pass<S, MT, PF, V2, F>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)(160 * 1024));
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    k_pass<S, MT, PF, V2, F><<<dim3(nwg), dim3(256), lds, st>>>(a);
    return hipGetLastError();
}

// Rows per tile of the generic pass, 32 F: the narrow instance takes F = 4
// (S <= 8) or 2 (S <= 16) when the tile's columns fit its prefetch
// registers (ncols * 32 F <= 256 * kNarrowPF) and the step-1 tiles fit.
int pass_f(int S, const PassArgs &a)
{
    if (!pass_narrow(a) || getenv("ORTH_PASS_TILE32")) return 1;
    for (int F = S <= 8 ? 4 : S <= 16 ? 2 : 1; F > 1; F >>= 1)
        if (a.ncols * kPT * F <= 256 * kNarrowPF && pass_lds_bytes(a, F) != 0) return F;
    return 1;
}

int pass_rows(int S, const PassArgs &a)
{
    if (S == 16 && pass16_mt(a) > 0 && !getenv("ORTH_GENERIC_PASS")) return kPT;  // k_pass16
    return kPT * pass_f(S, a);
}

// Two-row (16-byte) loads: even leading dimension and row count, 16-byte
// aligned slab.
bool pass_v2_ok(const PassArgs &a)
{
    return a.ldX % 2 == 0 && a.m % 2 == 0 && (uintptr_t)a.X % 16 == 0 &&
           !getenv("ORTH_PASS_LOAD8");
}

template <int S, int F>
hipError_t launch_pass_n(const PassArgs &a, size_t lds, int nwg, hipStream_t st)
{
    return pass_v2_ok(a) ? launch_pass_v<S, 4, kNarrowPF, true, F>(a, lds, nwg, st)
                         : launch_pass_v<S, 4, kNarrowPF, false, F>(a, lds, nwg, st);
}

template <int S>
hipError_t launch_pass_t(const PassArgs &a, int nwg, hipStream_t st)
{
    const int F = pass_f(S, a);
    const size_t lds = pass_lds_bytes(a, F);
    if (lds == 0 || a.rows_per % (kPT * F) != 0) return hipErrorInvalidValue;
    if (pass_narrow(a)) {
        if constexpr (S <= 8)
            if (F == 4) return launch_pass_n<S, 4>(a, lds, nwg, st);
        if constexpr (S <= 16)
            if (F == 2) return launch_pass_n<S, 2>(a, lds, nwg, st);
        return launch_pass_n<S, 1>(a, lds, nwg, st);
    }
    return launch_pass_v<S, kPassMaxTiles, kPF>(a, lds, nwg, st);
}

int pass_wg_per_cu(int S, const PassArgs &a, bool)
{
    const size_t lds = pass_lds_bytes(a, pass_f(S, a));
    if (lds == 0) return 1;
    // Register-limited residency (k_pass16 and the wide generic pass: one
    // workgroup per CU).
    const bool p16 = S == 16 && pass16_mt(a) > 0 && !getenv("ORTH_GENERIC_PASS");
    const int by_regs = p16 ? 1 : pass_narrow(a) ? pass_waves(S, 4) : pass_waves(S, kPassMaxTiles);
    const int by_lds = (int)std::max<size_t>(1, (160 * 1024) / lds);
    return std::max(1, std::min(by_regs, by_lds));
}

hipError_t launch_pass(int S, const PassArgs &a, int nwg, hipStream_t st)
{
    if (S == 16 && pass16_mt(a) > 0 && !getenv("ORTH_GENERIC_PASS")) {
        const size_t lds = pass_lds_bytes(a);
        if (lds == 0) return hipErrorInvalidValue;
        return launch_pass16(a, lds, nwg, st);
    }
    switch (S) {
    case 4: return launch_pass_t<4>(a, nwg, st);
    case 8: return launch_pass_t<8>(a, nwg, st);
    case 16: return launch_pass_t<16>(a, nwg, st);
    case 32: return launch_pass_t<32>(a, nwg, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace orth
