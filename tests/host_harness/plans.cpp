// Host-harness driver: runs the library's schedules for every column count
// and many block widths with the plan functions of the built library
// (liborth_hip.so, loaded at run time) in place of the stand-in's, kernels
// still doing nothing.  Every call must be accepted, and every fused pass must
// get a row chunk that its plan can tile.
#include <dlfcn.h>
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <stdlib.h>

#include <vector>

#include "orth_ext.h"
#include "orth_kernels.h"
#include "orth_scratch.h"

hipError_t stub_launch(hipStream_t s);

static int (*real_rows)(int, const orth::PassArgs &);
static int (*real_wg)(int, const orth::PassArgs &, bool);
static long passes = 0;

namespace orth {
int pass_rows(int S, const PassArgs &a) { return real_rows(S, a); }
int pass_wg_per_cu(int S, const PassArgs &a, bool tail) { return real_wg(S, a, tail); }
hipError_t launch_pass(int S, const PassArgs &a, int nwg, hipStream_t st)
{
    passes++;
    const int rows = real_rows(S, a);
    if (rows <= 0 || a.rows_per % rows != 0 || (int64_t)nwg * a.rows_per < a.m)
        return hipErrorInvalidValue;
    return stub_launch(st);
}
}  // namespace orth

int main(int argc, char **argv)
{
    void *lib = argc > 1 ? dlopen(argv[1], RTLD_NOW | RTLD_LOCAL) : nullptr;
    if (!lib) {
        printf("cannot load the library: %s\n", dlerror());
        return 2;
    }
    real_rows = (decltype(real_rows))dlsym(lib, "_ZN4orth9pass_rowsEiRKNS_8PassArgsE");
    real_wg = (decltype(real_wg))dlsym(lib, "_ZN4orth14pass_wg_per_cuEiRKNS_8PassArgsEb");
    if (!real_rows || !real_wg) {
        printf("plan functions not found\n");
        return 2;
    }
    // Kernels do nothing, so X is an address that is never read.
    double *X = (double *)(uintptr_t)(1 << 20), *R = nullptr;
    const int nmax = 530;
    hipMalloc(&R, (size_t)nmax * nmax * sizeof(double));
    // Fixed scratch of the size the allocation-free form has (48 MiB).
    using namespace orth;
    std::vector<double> store((size_t)6 << 20);
    Scratch sc;
    double *q = store.data();
    auto take = [&](size_t n) {
        double *p = q;
        q += (n + 31) & ~(size_t)31;
        return p;
    };
    sc.stash = take(scratch_stash_need());
    sc.status_d = (int *)take(32);
    sc.tickets = (int *)take(kTailTickets / 2);
    sc.P_n = scratch_p_need(512);
    sc.P[0] = take(sc.P_n);
    sc.P[1] = take(sc.P_n);
    sc.Rd_n = scratch_r_need(512);
    sc.Rd = take(sc.Rd_n);
    sc.Cbuf_n = scratch_cbuf_need(512);
    sc.Cbuf = take(sc.Cbuf_n);
    sc.part = q;
    sc.part_n = store.data() + store.size() - q;
    sc.fixed = true;

    int bad = 0, calls = 0;
    auto expect = [&](const char *what, int variant, int64_t m, int64_t n, int64_t s, int rc) {
        calls++;
        if (rc == 0) return;
        if (bad++ < 20)
            printf("%s variant %d m %lld n %lld s %lld: rc %d\n", what, variant, (long long)m,
                   (long long)n, (long long)s, rc);
    };
    for (int s : {1, 2, 3, 4, 5, 7, 8, 9, 10, 13, 16, 17, 20, 25, 31, 32})
        for (int n = s; n <= nmax; n++) {
            if (s < 3 && n > 40 && n < 250 && n % 16 > 1) continue;  // (time)
            for (int64_t m : {(int64_t)n + 3, (int64_t)40000, (int64_t)1 << 22})
                for (int variant = ORTH_P1S; variant <= ORTH_P2S; variant++) {
                    if (s < 3 && m != 40000) continue;
                    expect("device", variant, m, n, s,
                           orth_bcgs_device(variant, m, n, s, X, m, R, n, nullptr));
                    if (n <= 512 && m == 40000)
                        expect("fixed scratch", variant, m, n, s,
                               run_on_fixed_scratch(variant, m, n, s, X, m, R, n, nullptr, sc,
                                                    256, nullptr));
                    if (s == 16 && variant == ORTH_P1S)
                        expect("mixed", variant, m, n, s,
                               orth_bcgs_mixed_device(variant, ORTH_PREC_FP64, m, n, s,
                                                      (const float *)X, m, X, m, R, n, nullptr));
                }
        }
    orth_release();
    printf("calls %d, fused passes %ld, refused %d\n", calls, passes, bad);
    return bad ? 1 : 0;
}
