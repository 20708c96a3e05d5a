// The dispatch of the FP64 fused passes: block widths up to 16 run the tile
// pass (orth_tpass.h), wider ones the wide-block pass (orth_wpass.h).
#include "orth_kernels.h"

namespace orth {

int pass_rows(int S, const PassArgs &a)
{
    return S == kMaxS ? wpass_rows(S, a) : tpass_rows(S, a);
}

int pass_wg_per_cu(int S, const PassArgs &a, bool)
{
    return S == kMaxS ? wpass_wg_per_cu(S, a) : tpass_wg_per_cu(S, a);
}

hipError_t launch_pass(int S, const PassArgs &a, int nwg, hipStream_t st)
{
    return S == kMaxS ? launch_wpass(S, a, nwg, st) : launch_tpass(S, a, nwg, st);
}

}  // namespace orth
