// The resize launcher of csrc/transforms.hip against a runtime that refuses to raise a kernel's LDS limit, on the CPU: the runtime's entry points below
// stand in for libamdhip64's.  Built and run by tests/test_host_resize.py.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "../include/rtvla.h"

static bool refuse;
static int launches;
static size_t last_smem;
static hipError_t last_error = hipSuccess;
static hipError_t set(hipError_t e) { if (e != hipSuccess) last_error = e; return e; }

extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return set(refuse ? hipErrorInvalidValue : hipSuccess); }
hipError_t hipGetLastError() { const hipError_t e = last_error; last_error = hipSuccess; return e; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t smem, hipStream_t) { ++launches; last_smem = smem; return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t smem, hipStream_t) { last_smem = smem; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t* smem, hipStream_t* s) { *smem = last_smem; *s = nullptr; return hipSuccess; }
void** __hipRegisterFatBinary(const void*) { static void* handle; return &handle; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipUnregisterFatBinary(void**) {}
}

int main() {
    char frame[64], out[64];                                   // never read: nothing is launched
    int failures = 0;
    size_t smem[2];
    for (int k = 0; k < 2; ++k) {                              // refused first: what was granted once is not asked for again
        refuse = k == 0;
        launches = 0;
        const int rc = rtvla_preprocess_frame(frame, 1, 480, 640, out, nullptr);
        smem[k] = last_smem;
        if (rc != RTVLA_OK || launches != 1 || last_error != hipSuccess) { ++failures; fprintf(stderr, "limit %s: status %d, %d launches, pending error %d\n", refuse ? "refused" : "raised", rc, launches, (int)last_error); }
    }
    if (smem[0] >= smem[1]) { ++failures; fprintf(stderr, "the frame was not staged with the limit raised: %zu bytes of LDS against %zu\n", smem[1], smem[0]); }
    printf(failures ? "%d check(s) failed\n" : "all checks passed\n", failures);
    return failures != 0;
}
