// Host-harness driver: where R and the status of a call go, by the kind of
// memory the caller passes.  A kernel may write only to memory of the current
// device, to managed memory and to host memory whose device address is its
// host address; everything else goes through copies.
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "orth_ext.h"
#include "orth_kernels.h"

hipError_t stub_launch(hipStream_t s);

static const int N = 24;
static double mem[5][N * N];
static hipPointerAttribute_t kind[5];
static const void *kernel_dst;
static bool copied;

hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    memset(a, 0, sizeof(*a));
    for (int k = 0; k < 5; k++) {
        const char *b = (const char *)mem[k], *c = (const char *)p;
        if (c < b || c >= b + sizeof(mem[k])) continue;
        *a = kind[k];
        if (a->devicePointer) a->devicePointer = (char *)a->devicePointer + (c - b);
    }
    return hipSuccess;
}

hipError_t hipMemcpy2DAsync(void *d, size_t, const void *, size_t, size_t, size_t, hipMemcpyKind,
                            hipStream_t)
{
    for (int k = 0; k < 5; k++)
        if ((char *)d >= (char *)mem[k] && (char *)d < (char *)mem[k] + sizeof(mem[k])) copied = true;
    return hipSuccess;
}

namespace orth {
hipError_t launch_small(const SmallArgs &a, hipStream_t st)
{
    if (a.op == OP_FINISH && a.Rdst) kernel_dst = a.Rdst;
    return stub_launch(st);
}
}  // namespace orth

int main()
{
    const char *names[5] = {"current device", "another device", "managed", "pinned host",
                            "host mapped elsewhere"};
    const bool kernel[5] = {true, false, true, true, false};
    kind[0].type = kind[1].type = hipMemoryTypeDevice;
    kind[1].device = 1;
    kind[2].type = hipMemoryTypeManaged;
    kind[3].type = kind[4].type = hipMemoryTypeHost;
    for (int k = 0; k < 5; k++) kind[k].devicePointer = mem[k];
    kind[4].devicePointer = (char *)mem[4] + ((size_t)1 << 40);
    int bad = 0;
    double *X = (double *)(uintptr_t)(1 << 20);  // never read
    for (int k = 0; k < 5; k++) {
        kernel_dst = nullptr;
        copied = false;
        const int rc = orth_bcgs_device(ORTH_P1S, 1000, N, 8, X, 1000, mem[k], N, nullptr);
        const bool ok = rc == 0 && (kernel_dst == mem[k]) == kernel[k] && copied == !kernel[k];
        printf("%s: rc %d, %s%s\n", names[k], rc, kernel_dst ? "kernel" : copied ? "copies" : "none",
               ok ? "" : "  UNEXPECTED");
        bad += !ok;
    }
    orth_release();
    return bad;
}
