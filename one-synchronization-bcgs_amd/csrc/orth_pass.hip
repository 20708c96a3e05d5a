// The fused pass for block widths 17 to 32 (256 threads), and the dispatch of
// the FP64 passes: every narrower block runs the tile pass (orth_tpass.h).
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

// One workgroup per CU (up to 512 registers per lane).  MT: projection tiles
// per wave, PF: prefetch registers per thread.  V2: every lane moves two
// consecutive rows with one 16-byte load (even ldX and m, 16-byte aligned
// slab).
template <int MT, int PF, bool V2>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_pass(PassArgs a)
{
    constexpr int S = kMaxS, TS = kPT, PLD = TS + 1;
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

// The narrow instance: at most kNarrowCols columns and 4 projection tiles
// per wave.
constexpr int kNarrowCols = 160;
constexpr int kNarrowPF = kNarrowCols * kPT / 256;

static bool pass_narrow(const PassArgs &a)
{
    const int Ma = (a.na + 15) / 16, Nb = (a.nb + 15) / 16;
    return a.ncols <= kNarrowCols && (a.na == 0 || Ma * Nb <= 4 * 4);
}

// Two-row (16-byte) loads: even leading dimension and row count, 16-byte
// aligned slab.
static bool pass_v2_ok(const PassArgs &a)
{
    return a.ldX % 2 == 0 && a.m % 2 == 0 && (uintptr_t)a.X % 16 == 0;
}

template <int MT, int PF, bool V2>
static hipError_t launch_pass_v(const PassArgs &a, size_t lds, int nwg, hipStream_t st)
{
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void *)k_pass<MT, PF, V2>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)(160 * 1024));
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    k_pass<MT, PF, V2><<<dim3(nwg), dim3(256), lds, st>>>(a);
    return hipGetLastError();
}

int pass_rows(int S, const PassArgs &a)
{
    const int ts = tpass_rows(S, a);
    return ts > 0 ? ts : kPT;
}

int pass_wg_per_cu(int S, const PassArgs &a, bool)
{
    return tpass_rows(S, a) > 0 ? tpass_wg_per_cu(S, a) : 1;
}

hipError_t launch_pass(int S, const PassArgs &a, int nwg, hipStream_t st)
{
    if (tpass_rows(S, a) > 0) return launch_tpass(S, a, nwg, st);
    const size_t lds = pass_lds_bytes(a);
    if (S != kMaxS || lds == 0 || a.rows_per % kPT != 0) return hipErrorInvalidValue;
    if (!pass_narrow(a)) return launch_pass_v<kPassMaxTiles, kPF, false>(a, lds, nwg, st);
    return pass_v2_ok(a) ? launch_pass_v<4, kNarrowPF, true>(a, lds, nwg, st)
                         : launch_pass_v<4, kNarrowPF, false>(a, lds, nwg, st);
}

}  // namespace orth
