// Plan and launch of the wide-block pass (orth_wpass.h).
#include "orth_wpass.h"

#include <algorithm>

#include "orth_kernels.h"

namespace orth {

namespace {

struct WpPlan {
    int nw = 0;  // waves per workgroup, 0: the wide-block pass does not apply
    int ts = 0;  // rows per tile
    int wl = 0;  // columns of a buffer
    int zn = 0;  // 16-column tiles of Z in use (2 per group)
    int nb = 0;  // N-tiles of the projection (2 or 4)
    int bsh = 0;  // columns the first N-tile starts before b0
};

// LDS bytes: two buffers, partial Z tiles, one group's solve operands and the
// second group's (sequential form: its 32 x 32 coefficients).
template <int NW, int TS, int ZN>
constexpr size_t lds_w(int wl)
{
    return (size_t)(2 * wl * TS + WpZ<NW, TS, ZN>::Zs + ZN / 2 * 1024) * sizeof(double);
}

// Up to 256 columns two workgroups of 4 waves share a CU (80 KB each), which
// takes as many rows per tile as fit, fewer where the slab would otherwise
// leave workgroups without a tile (2 on each of 256 CUs); above, one
// workgroup of 8 waves holds it.
constexpr size_t kLds = 160 * 1024;

template <int NW, int TS>
bool fits(const WpPlan &p)
{
    return (p.zn == 2 ? lds_w<NW, TS, 2>(p.wl) : lds_w<NW, TS, 4>(p.wl)) <= kLds * NW / 8;
}

WpPlan plan(int S, const PassArgs &a)
{
    WpPlan p;
    if (S != kMaxS || a.X32 || a.n1 != kWpN1 || a.ncols > kWpassMaxCols || a.nb > 2 * kMaxS) return p;
    for (int g = 0; g < a.ngrp; g++)
        if (a.g[g].w > kMaxS || a.g[g].zoff != kMaxS * g || a.g[g].t0 + a.g[g].w > a.ncols ||
            (a.seq && g == 1 && a.g[g].T))
            return p;
    p.zn = a.ngrp > 1 ? 4 : 2;
    p.nb = a.nb > 32 ? 4 : 2;
    int wl = std::max(a.ncols, a.k1);
    if (a.na > 0) wl = std::max(wl, std::max(a.a0 + (a.na + 15) / 16 * 16, 16 * p.nb));
    p.wl = wl = (wl + 15) / 16 * 16;
    if (a.na > 0) p.bsh = std::max(0, a.b0 + 16 * p.nb - wl);
    p.nw = 4;
    if (wl <= 64 && !a.seq && a.m >= 64 * 512 && fits<4, 64>(p)) {
        p.ts = 64;
    } else if (wl <= 128 && a.m >= 32 * 512 && fits<4, 32>(p)) {
        p.ts = 32;
    } else if (wl <= 256 && fits<4, 16>(p)) {
        p.ts = 16;
    } else {
        p.nw = fits<8, 16>(p) ? 8 : 0;
        p.ts = p.nw ? 16 : 0;
    }
    return p;
}

template <int NW, int TS, int NB, int ZN, int MT, bool SEQ>
hipError_t launch_t(const PassArgs &a, int nwg, hipStream_t st)
{
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void *)k_wpass<NW, TS, NB, ZN, MT, SEQ>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)kLds);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    k_wpass<NW, TS, NB, ZN, MT, SEQ>
        <<<dim3(nwg), dim3(64 * NW), lds_w<NW, TS, ZN>(a.wl), st>>>(a);
    return hipGetLastError();
}

template <int NW, int TS, int MT>
hipError_t launch_n(const PassArgs &a, const WpPlan &p, int nwg, hipStream_t st)
{
    if (a.seq && a.ngrp > 1) {
        if constexpr (TS == 64)  // (not planned: its registers spill)
            return hipErrorInvalidValue;
        else
            return p.nb == 2 ? launch_t<NW, TS, 2, 4, MT, true>(a, nwg, st)
                             : launch_t<NW, TS, 4, 4, MT, true>(a, nwg, st);
    }
    if (p.zn == 2)
        return p.nb == 2 ? launch_t<NW, TS, 2, 2, MT, false>(a, nwg, st)
                         : launch_t<NW, TS, 4, 2, MT, false>(a, nwg, st);
    return p.nb == 2 ? launch_t<NW, TS, 2, 4, MT, false>(a, nwg, st)
                     : launch_t<NW, TS, 4, 4, MT, false>(a, nwg, st);
}

}  // namespace

int wpass_rows(int S, const PassArgs &a) { return plan(S, a).ts; }

int wpass_wg_per_cu(int S, const PassArgs &a) { return plan(S, a).nw == 8 ? 1 : 2; }

hipError_t launch_wpass(int S, const PassArgs &a0, int nwg, hipStream_t st)
{
    const WpPlan p = plan(S, a0);
    if (p.nw == 0 || a0.rows_per % p.ts != 0) return hipErrorInvalidValue;
    PassArgs a = a0;
    a.wl = p.wl;
    a.bsh = p.bsh;
    // The sequential form's last block: its own columns are no operands.
    if (a.seq && a.ngrp == 1) a.k1 = std::min(a.k1, a.g[0].t0);
    if (p.nw == 8) return launch_n<8, 16, 4>(a, p, nwg, st);
    switch (p.ts) {
    case 16: return launch_n<4, 16, 4>(a, p, nwg, st);
    case 32: return launch_n<4, 32, 2>(a, p, nwg, st);
    case 64: return launch_n<4, 64, 1>(a, p, nwg, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace orth
