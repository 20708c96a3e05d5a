// Plan and launch of the tile pass (orth_tpass.h).
#include "orth_tpass.h"

#include <algorithm>

#include "orth_kernels.h"

namespace orth {

namespace {

struct TpPlan {
    int nw = 0;   // waves per workgroup, 0: the tile pass does not apply
    int ts = 0;   // rows per tile
    int wl = 0;   // columns of a buffer
    int bsh = 0;  // columns the first N-tile of the projection starts before b0
};

// Block widths up to 16, FP64 columns, at most kTpassMaxCols of them.
//
// Rows per tile: two workgroups share a CU, so a buffer of TS rows takes
// TS wl <= kTpBuf doubles (16-row tiles: up to 256 columns); fewer where the
// slab would otherwise leave workgroups without a tile (2 on each of 256
// CUs).  A pass without a projection over more than 128 columns of a slab
// that no cache holds has little to compute and streams better in 256-byte
// runs: 32-row tiles, one workgroup of 16 waves per CU (2^24 x 256: 8.2
// against 9.2 ms; with a projection the same form takes 8.5 / 8.8 / 11.1 ms
// at 144 / 192 / 256 columns where two workgroups take 7.6 / 8.8 / 11.1).
// Over 256 columns the buffers need a whole CU.
constexpr int64_t kTpCached = 256 << 20;  // bytes of the last-level cache

TpPlan plan(int S, const PassArgs &a)
{
    TpPlan p;
    if (S > 16 || a.n1 > 32) return p;
    // Mixed form: at most 32 raw columns, none of them a step-1 operand.
    if (a.X32 && (a.n1 != 32 || a.seq || a.raw0 < a.k1 || a.ncols - a.raw0 > 32)) return p;
    int wl = std::max(a.ncols, a.k1);
    if (a.na > 0) {
        const int Ma = (a.na + 15) / 16, Nb = (a.nb + 15) / 16;
        if (Nb > a.n1 / 16) return p;
        wl = std::max(wl, std::max(a.a0 + 16 * Ma, 16 * Nb));
        // The N-tiles end with the buffer: no padding columns for them.
        wl = (wl + 15) / 16 * 16;
        p.bsh = std::max(0, a.b0 + 16 * Nb - wl);
    }
    wl = (wl + 15) / 16 * 16;
    // A projection on a block at the slab's end (the intra-block QR) pads its
    // M-tile past the last column.
    if (a.ncols > kTpassMaxCols || wl > kTpassMaxCols + 16) return p;
    for (int g = 0; g < a.ngrp; g++)
        if (a.g[g].t0 + a.g[g].w > a.ncols || a.g[g].zoff % 4 != 0 ||
            a.g[g].zoff / 16 != (a.g[g].zoff + a.g[g].w - 1) / 16)
            return p;
    p.wl = wl;
    p.nw = 8;
    p.ts = 128;
    while (p.ts > 16 && (p.ts * wl > kTpBuf || a.m < (int64_t)p.ts * 512)) p.ts >>= 1;
    if (wl > 256) {
        p.nw = 16;
    } else if (wl > 128 && a.na == 0 && a.m * wl * 8 > kTpCached) {
        p.nw = 16;
        p.ts = 32;
    }
    return p;
}

// Doubles beside the buffers: partial Z tiles, the sequential form's 16 x 16
// coefficients.
template <int NW, int TS, int ZN>
size_t lds_t(int wl, int seq)
{
    return (size_t)(2 * wl * TS + TpZ<NW, TS, ZN, false>::Zs + (seq ? 256 : 0)) * sizeof(double);
}

template <int NW, int TS, int NB, int ZN, int MT, bool WIDE, bool SEQ, bool MIX = false>
hipError_t launch_t(const PassArgs &a, int nwg, hipStream_t st)
{
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e =
            hipFuncSetAttribute((const void *)k_tpass<NW, TS, NB, ZN, MT, WIDE, SEQ, MIX>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)(160 * 1024));
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    k_tpass<NW, TS, NB, ZN, MT, WIDE, SEQ, MIX>
        <<<dim3(nwg), dim3(64 * NW), lds_t<NW, TS, ZN>(a.wl, SEQ), st>>>(a);
    return hipGetLastError();
}

template <int NW, int TS, int MT, bool WIDE, bool SEQ>
hipError_t launch_n(const PassArgs &a, int nwg, hipStream_t st)
{
    if constexpr (!WIDE && !SEQ) {
        if (a.X32)
            return a.nb > 16 ? launch_t<NW, TS, 2, 2, MT, false, false, true>(a, nwg, st)
                             : launch_t<NW, TS, 1, 2, MT, false, false, true>(a, nwg, st);
    }
    if (a.X32) return hipErrorInvalidValue;
    if (a.n1 <= 16) return launch_t<NW, TS, 1, 1, MT, WIDE, SEQ>(a, nwg, st);
    return a.nb > 16 ? launch_t<NW, TS, 2, 2, MT, WIDE, SEQ>(a, nwg, st)
                     : launch_t<NW, TS, 1, 2, MT, WIDE, SEQ>(a, nwg, st);
}

template <bool SEQ>
hipError_t launch_s(const PassArgs &a, const TpPlan &p, int nwg, hipStream_t st)
{
    if (p.nw == 16)
        return a.wl > 256 ? launch_n<16, 16, 2, true, SEQ>(a, nwg, st)
                          : launch_n<16, 32, 1, false, SEQ>(a, nwg, st);
    switch (p.ts) {
    case 16:
        return a.na > 128 ? launch_n<8, 16, 2, false, SEQ>(a, nwg, st)
                          : launch_n<8, 16, 1, false, SEQ>(a, nwg, st);
    // At most 128 columns: one M-tile per wave.
    case 32: return launch_n<8, 32, 1, false, SEQ>(a, nwg, st);
    case 64: return launch_n<8, 64, 1, false, SEQ>(a, nwg, st);
    case 128: return launch_n<8, 128, 1, false, SEQ>(a, nwg, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

int tpass_rows(int S, const PassArgs &a) { return plan(S, a).ts; }

int tpass_wg_per_cu(int S, const PassArgs &a)
{
    const TpPlan p = plan(S, a);
    return p.nw == 16 ? 1 : 2;
}

hipError_t launch_tpass(int S, const PassArgs &a0, int nwg, hipStream_t st)
{
    const TpPlan p = plan(S, a0);
    if (p.nw == 0 || a0.rows_per % p.ts != 0) return hipErrorInvalidValue;
    PassArgs a = a0;
    a.wl = p.wl;
    a.bsh = p.bsh;
    return a.seq ? launch_s<true>(a, p, nwg, st) : launch_s<false>(a, p, nwg, st);
}

}  // namespace orth
