// How many timings the library makes before a first call on a lattice, on a
// stand-in for the HIP runtime: Nt Nx Ny Nz, prints those of the first quality
// check and of the first FP64 run, less those of the second of each.
#include "hip_stand_in.h"

int main(int argc, char **argv)
{
    void *const lib = argc > 5 ? dlopen(argv[1], RTLD_NOW | RTLD_LOCAL) : nullptr;
    if (!lib) return 2;
    SYM(gf_stats_create);
    SYM(gf_stats_quality);
    SYM(gf_run_mixed);
    gf_lattice lat{{std::atoi(argv[2]), std::atoi(argv[3]), std::atoi(argv[4]), std::atoi(argv[5])}, GF_F64,
                   GF_LAYOUT_PATTERN18};
    double links = 0, gff = 0, theta = 0;
    gf_stats *st = nullptr;
    gf_run_result r;
    if (gf_stats_create(lat.dims, GF_LANDAU, GF_CRIT_AVERAGE, &st) != GF_OK) return 2;
    int quality = 0, run = 0;
    for (int sign = 1; sign >= -1; sign -= 2) {
        timings = 0;
        if (gf_stats_quality(st, &lat, &links, &gff, &theta, nullptr) != GF_OK) return 2;
        quality += sign * timings;
        timings = 0;
        if (gf_run_mixed(&lat, &links, GF_MAG, 1.7f, 1e-6f, 1e-12f, 1, GF_MIXED_FP64, 25, 5, 100, &r, nullptr) != GF_OK)
            return 2;
        run += sign * timings;
    }
    std::printf("quality %d run %d\n", quality, run);
    return 0;
}
