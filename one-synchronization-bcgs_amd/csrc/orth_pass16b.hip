// Plan and launch of the 512-thread s = 16 pass (orth_pass16b.h), FP64 form.
#include "orth_kernels.h"

#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "orth_pass16b.h"

namespace orth {

int pass16b_rows(const PassArgs &a)
{
    for (int f = 8; f >= 1; f >>= 1) {
        const int ts = 32 * f;
        if ((int64_t)a.wl * (ts + 1) <= kBTile && a.ncols * ts <= kBPF * kB) return ts;
    }
    return 0;
}

size_t pass16b_lds_bytes(const PassArgs &a, int ts)
{
    return ((size_t)a.wl * (ts + 1) + 1024) * sizeof(double);
}

// 16-byte loads when the slab allows them: even leading dimension and a
// 16-byte aligned base (rows_per and the first row of every chunk are even).
template <int MT, int NB, int F, bool EARLY = false>
hipError_t launch_pass16b_t(const PassArgs &a, size_t lds, int nwg, hipStream_t st)
{
    const bool v2 = (a.ldX % 2 == 0) && ((uintptr_t)a.X % 16 == 0) && (a.rows_per % 2 == 0);
    return v2 ? launch_pass16b_v<MT, NB, F, EARLY, true>(a, lds, nwg, st)
              : launch_pass16b_v<MT, NB, F, EARLY, false>(a, lds, nwg, st);
}

// Passes without a projection.
hipError_t launch_pass16b_noproj(const PassArgs &a, int ts, size_t lds, int nwg, hipStream_t st)
{
    switch (ts) {
    case 32: return launch_pass16b_t<1, 1, 1, true>(a, lds, nwg, st);
    case 64: return launch_pass16b_t<1, 1, 2, true>(a, lds, nwg, st);
    case 128: return launch_pass16b_t<1, 1, 4, true>(a, lds, nwg, st);
    case 256: return launch_pass16b_t<1, 1, 8, true>(a, lds, nwg, st);
    default: return hipErrorInvalidValue;
    }
}

// Only the (MT, F) pairs the plan can produce are instantiated: a tile of
// TS = 32 F rows holds at most 8192 / TS columns, so MT <= 4 / F.
template <int MT, int NB>
hipError_t launch_pass16b_f(const PassArgs &a, int ts, size_t lds, int nwg, hipStream_t st)
{
    switch (ts) {
    case 32: return launch_pass16b_t<MT, NB, 1>(a, lds, nwg, st);
    case 64:
        if constexpr (MT <= 2) return launch_pass16b_t<MT, NB, 2>(a, lds, nwg, st);
        break;
    case 128:
        if constexpr (MT == 1) return launch_pass16b_t<MT, NB, 4>(a, lds, nwg, st);
        break;
    case 256:
        if constexpr (MT == 1) return launch_pass16b_t<MT, NB, 8>(a, lds, nwg, st);
        break;
    default: break;
    }
    return hipErrorInvalidValue;
}

// Super-tile rows of the 512-thread s = 16 pass, or 0 when it does not apply.
int pass16b_plan(const PassArgs &a, int *mt, int *nb)
{
    if (a.n1 != 32 || (a.na > 0 && a.nb > 32)) return 0;
    const int ts = pass16b_rows(a);
    if (ts == 0) return 0;
    if (pass16b_lds_bytes(a, ts) > 160 * 1024) return 0;
    if (a.na > 0) {
        const int Ma = (a.na + 15) / 16;
        if (a.a0 + Ma * 16 > a.wl || a.b0 + ((a.nb + 15) / 16) * 16 > a.wl) return 0;
        *nb = a.nb > 16 ? 2 : 1;
        *mt = (Ma + (*nb == 2 ? 3 : 7)) / (*nb == 2 ? 4 : 8);
        if (*mt > 4) return 0;
    } else {
        *nb = 1;
        *mt = 1;
    }
    for (int g = 0; g < a.ngrp; g++)
        if (a.g[g].w > 16 || a.g[g].t0 + a.g[g].w > a.ncols) return 0;
    return ts;
}

hipError_t launch_pass16b(const PassArgs &a, int nwg, hipStream_t st)
{
    int mt = 0, nb = 0;
    const int ts = pass16b_plan(a, &mt, &nb);
    if (ts == 0) return hipErrorInvalidValue;
    const size_t lds = pass16b_lds_bytes(a, ts);
    if (a.na == 0) return launch_pass16b_noproj(a, ts, lds, nwg, st);
#define ORTH_P16B(M)                                                                 \
    case M:                                                                          \
        return nb == 2 ? launch_pass16b_f<M, 2>(a, ts, lds, nwg, st)                \
                       : launch_pass16b_f<M, 1>(a, ts, lds, nwg, st);
    switch (mt) {
        ORTH_P16B(1)
        ORTH_P16B(2)
        ORTH_P16B(3)
        ORTH_P16B(4)
    default: return hipErrorInvalidValue;
    }
#undef ORTH_P16B
}

}  // namespace orth
