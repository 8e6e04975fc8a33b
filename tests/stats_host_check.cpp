// A gauge-quality handle's host side on a stand-in for the HIP runtime.
#include "hip_stand_in.h"

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
