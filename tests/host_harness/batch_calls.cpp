// Host-harness driver: what the first calls for one batch launch.  A batch met
// for the first time runs directly; when the next call is for the same batch
// it is captured and replayed at once; from then on it is replayed.
#include <hip/hip_runtime.h>
#include <stdio.h>

#include <vector>

#include "orth_ext.h"
#include "orth_kernels.h"

hipError_t stub_launch(hipStream_t s);
hipError_t stub_hipGraphLaunch(hipGraphExec_t x, hipStream_t s);
extern int g_stub_failures;

static int direct, captured, replays;

hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s)
{
    replays++;
    return stub_hipGraphLaunch(x, s);
}

namespace orth {
hipError_t launch_pass(int, const PassArgs &, int, hipStream_t st)
{
    hipStreamCaptureStatus cs;
    hipStreamIsCapturing(st, &cs);
    (cs == hipStreamCaptureStatusActive ? captured : direct)++;
    return stub_launch(st);
}
}  // namespace orth

int main()
{
    std::vector<int64_t> m, n, s;
    std::vector<double *> X, R;
    for (int i = 0; i < 12; i++) {
        m.push_back(4096 + 100 * i);
        n.push_back(i % 2 ? 32 : 64);
        s.push_back(8);
        double *x = nullptr, *r = nullptr;
        hipMalloc(&x, (size_t)m[i] * n[i] * 8);
        hipMalloc(&r, (size_t)n[i] * n[i] * 8);
        X.push_back(x);
        R.push_back(r);
    }
    int bad = 0;
    auto call = [&](const char *what, int count, bool d, bool c, bool g) {
        direct = captured = replays = 0;
        const int rc = orth_bcgs_batched_device(ORTH_P1S, count, m.data(), n.data(), s.data(), X.data(),
                                                m.data(), R.data(), n.data(), nullptr, 0, nullptr,
                                                nullptr);
        const bool ok = rc == 0 && (direct > 0) == d && (captured > 0) == c && (replays > 0) == g;
        printf("%s: rc %d, direct %d, captured %d, replays %d%s\n", what, rc, direct, captured,
               replays, ok ? "" : "  UNEXPECTED");
        bad += !ok;
    };
    call("first", 12, true, false, false);
    call("second", 12, false, true, true);
    call("third", 12, false, false, true);
    call("another batch", 6, true, false, false);
    call("the first again", 12, true, false, false);
    call("and again", 12, false, true, true);
    orth_release();
    for (double *p : X) hipFree(p);
    for (double *p : R) hipFree(p);
    return bad || g_stub_failures;
}
