// A gauge-quality handle's host side on a stand-in for the HIP runtime (the
// functions below take the place of libamdhip64's in this process): memory is
// the host's and not zeroed, fills wait on their stream until something runs
// that stream, and kernels are recorded but not run.
#include <dlfcn.h>

#include <cmath>
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
int launches = 0, unordered = 0, not_zero = 0;
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

int main(int argc, char **argv)
{
    void *const lib = argc > 1 ? dlopen(argv[1], RTLD_NOW | RTLD_LOCAL) : nullptr;
    if (!lib) {
        std::printf("no library: %s\n", dlerror());
        return 2;
    }
    SYM(gf_set_block_order);
    SYM(gf_stats_create);
    SYM(gf_stats_quality);
    SYM(gf_stats_destroy);
    gf_set_block_order(0, nullptr);  // nothing to tune
    const hipStream_t stream = (hipStream_t)(uintptr_t)64;  // a stream that the null stream does not wait for
    gf_lattice lat{{4, 4, 4, 8}, GF_F64, GF_LAYOUT_PATTERN18};
    double links = 0, gff = 0, theta = 0;
    gf_stats *st = nullptr;
    if (gf_stats_create(lat.dims, GF_LANDAU, GF_CRIT_AVERAGE, &st) != GF_OK) return 2;

    // a check whose kernel leaves no result, before and after one that does
    int stale = 0;
    for (int pass = 0; pass < 3; pass++) {
        write_result = pass == 1;
        if (gf_stats_quality(st, &lat, &links, &gff, &theta, stream) != GF_OK) return 2;
        if (!write_result && !(std::isnan(gff) && std::isnan(theta))) stale++;
    }
    gf_stats_destroy(st);
    std::printf("launches %d words %zu unordered %d not_zero %d stale %d\n", launches, words.size(), unordered, not_zero,
                stale);
    return 0;
}
