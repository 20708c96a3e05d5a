// Plan and launch of the double-buffered s = 16 pass (orth_pass16d.h), FP64
// form.
#include "orth_kernels.h"

#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "orth_pass16d.h"

namespace orth {

// The double-buffered s = 16 pass (orth_pass16d.h) with 32-row tiles: waves
// per workgroup (8: two workgroups per CU, when both buffers of two
// workgroups fit a CU's LDS; 16: one workgroup per CU, up to the whole
// 160 KB), or 0 when it does not apply.  It needs FP64 data with an even
// row count and leading dimension and a 16-byte aligned slab (16-byte loads
// of row pairs), the folded (non-sequential) step 1, and at least
// kPass16dMinCols columns: measured at m = 2^24, n = 256, it beats k_pass16b
// on the passes over 128 columns and more (by up to 0.8 ms each) and loses
// on the narrower ones, where k_pass16b runs two workgroups per CU with 64-
// to 256-row super-tiles (ORTH_PASS16D_MINCOLS overrides the bound).
constexpr int kPass16dMinCols = 128;

int pass16d_plan(const PassArgs &a, int *mt, int *nb, bool any_width, int min_cols)
{
    if (getenv("ORTH_PASS_REGPF")) return 0;
    if (a.n1 != 32 || a.seq || (a.na > 0 && a.nb > 32)) return 0;
    if (a.X32) {
        // Mixed form: at most 32 raw (FP32) columns, none of them a step-1
        // operand, a 16-column aligned frontier, no reduced-precision update.
        const int ndma = std::min(a.ncols, a.raw0);
        if (a.raw0 % 16 != 0 || a.ncols - ndma > 32 || ((a.k1 + 3) & ~3) > ndma) return 0;
        for (int g = 0; g < a.ngrp; g++)
            if (a.g[g].lp) return 0;
    }
    // Row pairs are loaded whole: an odd row count would read past the last
    // row of the last column.
    if (a.ldX % 2 != 0 || a.m % 2 != 0 || (uintptr_t)a.X % 16 != 0) return 0;
    int minc = any_width ? 1 : min_cols > 0 ? min_cols : kPass16dMinCols;
    if (const char *e = getenv("ORTH_PASS16D_MINCOLS")) minc = atoi(e);
    if (a.ncols < minc || a.ncols > a.wl) return 0;
    const bool force16 = getenv("ORTH_PASS16D_ONEWG") != nullptr;
    int nw = 0;
    if (!force16 && 2 * pass16d_lds(a.wl, 8) <= kDLds) nw = 8;
    else if (pass16d_lds(a.wl, 16) <= kDLds) nw = 16;
    if (nw == 0) return 0;
    const int ks = nw / 4;
    const int nks = a.k1 > 0 ? ((a.k1 + 3) & ~3) / 4 : 0;
    if ((nks + ks - 1) / ks > kDKq || (a.k1 > 0 && ((a.k1 + 3) & ~3) > a.wl)) return 0;
    // Each group's Z columns are one whole Z tile (zoff 0 or 16, distinct):
    // the wave that sums that tile solves the group.
    for (int g = 0; g < a.ngrp; g++)
        if (a.g[g].w > 16 || a.g[g].t0 + a.g[g].w > a.ncols || a.g[g].t0 % 16 != 0 ||
            a.g[g].t0 + 16 > a.wl || (a.g[g].zoff != 0 && a.g[g].zoff != 16))
            return 0;
    if (a.ngrp == 2 && a.g[0].zoff == a.g[1].zoff) return 0;
    *mt = 1;
    *nb = 1;
    if (a.na > 0) {
        const int Ma = (a.na + 15) / 16, Nb = (a.nb + 15) / 16;
        if (a.a0 + Ma * 16 > a.wl || a.b0 + Nb * 16 > a.wl) return 0;
        // The LDS bound (wl <= 128 with 8 waves, <= 256 with 16) keeps Ma
        // within one M-tile per wave.
        *mt = (Ma + nw - 1) / nw;
        *nb = Nb;
        if (*mt > 1) return 0;
    }
    return nw;
}

template <int NW, int NB>
hipError_t launch_pass16d_t(const PassArgs &a, int nwg, hipStream_t st)
{
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void *)k_pass16d<NW, NB, 0>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)(160 * 1024));
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    const size_t lds = (size_t)pass16d_lds(a.wl, NW) * sizeof(double);
    k_pass16d<NW, NB, 0><<<dim3(nwg), dim3(64 * NW), lds, st>>>(a);
    return hipGetLastError();
}

template <int NW>
hipError_t launch_pass16d_nw(const PassArgs &a, int mt, int nb, int nwg, hipStream_t st)
{
    if (mt != 1) return hipErrorInvalidValue;
    return nb == 2 ? launch_pass16d_t<NW, 2>(a, nwg, st) : launch_pass16d_t<NW, 1>(a, nwg, st);
}

hipError_t launch_pass16d(const PassArgs &a, int nw, int nb, int nwg, hipStream_t st)
{
    if ((nw != 8 && nw != 16) || a.rows_per % 32 != 0) return hipErrorInvalidValue;
    return nw == 16 ? launch_pass16d_nw<16>(a, 1, nb, nwg, st) : launch_pass16d_nw<8>(a, 1, nb, nwg, st);
}

}  // namespace orth
