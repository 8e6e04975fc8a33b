// A stand-in for the HIP runtime, for tests of the library's host side on the
// CPU: the functions below take the place of libamdhip64's in the test's
// process.  Memory is the host's and not zeroed, fills wait on their stream
// until something runs that stream, and kernels are counted but not run.
#pragma once
#include <dlfcn.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include <hip/hip_runtime_api.h>

#include "su3gf.h"

namespace {
struct Fill {
    void *p;
    int value;
    size_t n;
    hipStream_t s;
};
std::vector<Fill> fills;        // not yet run
std::vector<uint32_t *> words;  // device allocations of one 32-bit word
std::vector<double *> pinned;
int launches = 0, unordered = 0, not_zero = 0, timings = 0;
bool write_result = false;

void run_fills(hipStream_t s, bool all)
{
    std::vector<Fill> left;
    for (const Fill &f : fills) {
        if (all || f.s == s) std::memset(f.p, f.value, f.n);
        else left.push_back(f);
    }
    fills.swap(left);
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n)
{
    *p = std::malloc(n);
    std::memset(*p, 0xab, n);
    if (n == 4) words.push_back((uint32_t *)*p);
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    *p = std::malloc(n);
    for (size_t k = 0; k < n / sizeof(double); k++) ((double *)*p)[k] = 42.0;
    pinned.push_back((double *)*p);
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    std::free(p);
    return hipSuccess;
}
// of device memory: may return before it has run
hipError_t hipMemset(void *p, int value, size_t n)
{
    fills.push_back({p, value, n, nullptr});
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int value, size_t n, hipStream_t s)
{
    fills.push_back({p, value, n, s});
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    run_fills(s, false);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize()
{
    run_fills(nullptr, true);
    return hipSuccess;
}
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t)
{
    *p = std::calloc(n, 1);
    return hipSuccess;
}
hipError_t hipFreeAsync(void *p, hipStream_t)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(to, from, n);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e)
{
    *e = (hipEvent_t)std::malloc(1);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.0f;
    timings++;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
static dim3 cfg_grid, cfg_block;
static size_t cfg_lds;
static hipStream_t cfg_stream;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s)
{
    cfg_grid = grid;
    cfg_block = block;
    cfg_lds = lds;
    cfg_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s)
{
    *grid = cfg_grid;
    *block = cfg_block;
    *lds = cfg_lds;
    *s = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t s)
{
    launches++;
    run_fills(s, false);
    if (!fills.empty()) unordered++;  // on another stream, which nothing orders before this one
    for (const uint32_t *w : words)
        if (*w != 0) not_zero++;
    if (write_result)
        for (double *d : pinned) d[0] = d[1] = 1.0;
    return hipSuccess;
}
}  // extern "C"

#define SYM(name) const auto name = (decltype(&::name))dlsym(lib, #name)
