// The synchronization between passes (gfx950):
//
//  k_reduce        fixed-order sum of the projection partials (the in-kernel
//                  replacement of the reference's MPI_Allreduce)
//  k_reduce_small  the same sum and the small step after it in one launch
//  k_small         a small step on its own (orth_small.h)
#include "orth_kernels.h"

#include <algorithm>

#include "orth_device.h"
#include "orth_small.h"
#include "orth_tail.h"

namespace orth {

// Sums of the partials of EL elements in the fixed order of the in-pass tail
// (tail_group), by NT threads: thread (el, q) sums groups q, q + NT / EL, ...
// of element blockIdx.x * EL + el into red, then q == 0 adds the group sums in
// order.
template <int NT, int EL = 32>
static __device__ __forceinline__ double reduce_fixed_order(const double *__restrict__ part, int nwg,
                                                            int grp, int64_t E, double *red)
{
    const int el = threadIdx.x % EL, q = threadIdx.x / EL;
    const int64_t e = (int64_t)blockIdx.x * EL + el;
    const int ngrp = (nwg + grp - 1) / grp;
    if (e < E)
        for (int g = q; g < ngrp; g += NT / EL)
            red[EL * g + el] = part_range_sum(part, E, e, g * grp, min(nwg, g * grp + grp));
    __syncthreads();
    double t = 0.0;
    if (q == 0 && e < E) {
        t = red[el];
        for (int g = 1; g < ngrp; g++) t += red[EL * g + el];
    }
    return t;
}

__global__ __launch_bounds__(256) void k_reduce(const double *__restrict__ part, int nwg, int grp,
                                                int64_t na, int64_t E,
                                                double *__restrict__ out, int64_t ldo)
{
    __shared__ double red[kTailMaxGroups * 32];
    const double t = reduce_fixed_order<256>(part, nwg, grp, E, red);
    const int64_t e = (int64_t)blockIdx.x * 32 + (threadIdx.x & 31);
    if ((threadIdx.x >> 5) == 0 && e < E) {
        const int64_t i = e % na, j = e / na;
        out[i + j * ldo] = t;
    }
}

hipError_t launch_reduce(const double *part, int nwg, int64_t na, int64_t nb, double *out,
                         int64_t ldo, hipStream_t st)
{
    const int64_t E = na * nb;
    if (E <= 0) return hipSuccess;
    k_reduce<<<dim3((unsigned)((E + 31) / 32)), dim3(256), 0, st>>>(part, nwg, tail_group(nwg), na,
                                                                   E, out, ldo);
    return hipGetLastError();
}

// Block width template of a small step's LDS and registers.
static int small_width(const SmallArgs &a) { return a.S <= 16 ? 16 : 32; }

// k_reduce's fixed-order sum, then the small step in the last workgroup to
// finish (ticket counter, publication as in the in-pass tail).  32 threads for
// each of EL elements: a thread sums one group of partials (one memory round
// trip).  With 1024 threads the small step has 16 waves for its prefix Gram and
// its rows of R and C.
constexpr int kRS = 1024;
template <int W, int NT, int EL>
__global__ __launch_bounds__(NT) void k_reduce_small(const double *__restrict__ part, int nwg,
                                                     int grp, int64_t E, double *out,
                                                     int *ticket, SmallArgs sm)
{
    constexpr int N = small_lds<W>() > kTailMaxGroups * EL ? small_lds<W>() : kTailMaxGroups * EL;
    __shared__ double lds[N];
    __shared__ int last;
    const double t = reduce_fixed_order<NT, EL>(part, nwg, grp, E, lds);
    const int64_t e = (int64_t)blockIdx.x * EL + threadIdx.x % EL;
    if (threadIdx.x / EL == 0 && e < E) out[e] = t;
    if (!tail_ticket(ticket, (int)gridDim.x - 1, &last)) return;
    if (threadIdx.x == 0) *ticket = 0;
    small_step<W>(NT, sm, lds);
}

template <int W, int NT, int EL>
static hipError_t launch_rs(const double *part, int nwg, int64_t E, double *out, int *ticket,
                            const SmallArgs &sm, hipStream_t st)
{
    k_reduce_small<W, NT, EL><<<dim3((unsigned)((E + EL - 1) / EL)), dim3(NT), 0, st>>>(
        part, nwg, tail_group(nwg), E, out, ticket, sm);
    return hipGetLastError();
}

hipError_t launch_reduce_small(const double *part, int nwg, int64_t na, int64_t nb, double *out,
                               int *ticket, const SmallArgs &sm, hipStream_t st)
{
    const int64_t E = na * nb;
    if (E <= 0) return hipErrorInvalidValue;
    // A CholQR step has no prefix, so 16 waves of it only wait at each other's
    // barriers: 256 threads, 8 elements each workgroup, up to 128 elements
    // (blocks of 11).  BCGSI+ with 1024 / 256 threads, 4099 rows: 64 x 2 3.93 /
    // 3.60 ms, 64 x 4 2.04 / 1.90, 200 x 10 3.08 / 3.00; 256 x 16 even (2.90 /
    // 2.86, P-2S 1.83 / 1.84), 96 x 24 0.94 / 1.07.
    if (small_width(sm) > 16) return launch_rs<32, kRS, 32>(part, nwg, E, out, ticket, sm, st);
    return sm.op >= OP_CQR1 && sm.op <= OP_CQR3 && E <= 128
               ? launch_rs<16, 256, 8>(part, nwg, E, out, ticket, sm, st)
               : launch_rs<16, kRS, 32>(part, nwg, E, out, ticket, sm, st);
}

// ---------------------------------------------------------------------------
// Small-matrix steps on their own (one workgroup, FP64)
// ---------------------------------------------------------------------------

template <int W>
__global__ __launch_bounds__(kRS) void k_small(SmallArgs a)
{
    __shared__ double lds[small_lds<W>()];
    small_step<W>(kRS, a, lds);
}

// Start and end of a call in one launch each (a launch costs about 4.6 us in
// a full queue, and a fill or a strided copy of R moves at most a few
// hundred KB).
__global__ __launch_bounds__(256) void k_init(SmallArgs a)
{
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, n = (int64_t)gridDim.x * 256;
    for (int64_t i = t; i < a.m; i += n) a.R[i] = 0.0;
    for (int64_t i = t; i < a.nslot; i += n) a.Sig[i] = 0.0;
    if (t < 4) a.status[t] = 0;
    if (a.tickets && t < kTailTickets) a.tickets[t] = 0;
}

// Workgroup (x, j): rows 256 x .. 256 x + 255 of column j.
__global__ __launch_bounds__(256) void k_finish(SmallArgs a)
{
    const int j = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
    const int rows = min(a.c, (j / a.wb + 1) * a.wb);
    if (a.Rdst && i < rows) a.Rdst[i + j * a.ldRdst] = a.R[i + j * a.ldR];
    if (a.info && blockIdx.x == 0 && j == 0 && threadIdx.x < 2)
        a.info[threadIdx.x] = a.status[threadIdx.x];
}

hipError_t launch_small(const SmallArgs &a, hipStream_t st)
{
    if (a.op == OP_INIT) {
        const int64_t n = a.m > a.nslot ? a.m : a.nslot;
        k_init<<<dim3((unsigned)std::min<int64_t>((n + 255) / 256, 1024)), dim3(256), 0, st>>>(a);
        return hipGetLastError();
    }
    if (a.op == OP_FINISH) {
        k_finish<<<dim3((a.c + 255) / 256, a.c), dim3(256), 0, st>>>(a);
        return hipGetLastError();
    }
    if (small_width(a) == 16)
        k_small<16><<<dim3(1), dim3(kRS), 0, st>>>(a);
    else
        k_small<32><<<dim3(1), dim3(kRS), 0, st>>>(a);
    return hipGetLastError();
}

}  // namespace orth
