// su3gf_fast.hip -- sweep kernels of the fused-check drivers (FMA
// contraction, hardware rsqrt): theta/gff of the lattice are accumulated inside
// the sweep (odd sites after the odd update, even sites before the next even
// update, finished by the last block of each kernel), and the FP32 phase of the
// mixed-precision driver also accumulates each site's gauge transformation.
#include "su3gf_sweep.h"

namespace su3gf {
namespace fast {

template <typename R, int G, int S, int T, bool GA> static hipError_t launch_t(SweepArgs<R> a, hipStream_t s)
{
    const dim3 grid((unsigned)sweep_grid(a.g)), block(kBlock);
    // (GA: g's 12 floats per site stay in the cache too)
    a.keep = kept_links(a.g.Vh, (48 + (GA ? 12 : 0)) * (int64_t)sizeof(R) * a.g.V);
    if (a.keep < 4 * a.g.Vh) hipLaunchKernelGGL((k_sweep<R, G, GF_OR, S, false, T, GA, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((k_sweep<R, G, GF_OR, S, false, T, GA, false>), grid, block, 0, s, a);
    return hipGetLastError();
}

template <typename R, int G, int S, bool GA>
static hipError_t launch_theta(int theta, const SweepArgs<R> &a, hipStream_t s)
{
    switch (theta) {
    case 1: return launch_t<R, G, S, 1, GA>(a, s);
    case 2: return launch_t<R, G, S, 2, GA>(a, s);
    case 3:
        // the read-only pass does not touch g
        if (GA || !a.state) return hipErrorInvalidValue;
        return launch_t<R, G, S, 3, false>(a, s);
    default: return launch_t<R, G, S, 0, GA>(a, s);
    }
}

template <typename R, int S, bool GA>
static hipError_t launch_g(int gauge, int theta, const SweepArgs<R> &a, hipStream_t s)
{
    switch (gauge) {
    case GF_LANDAU: return launch_theta<R, GF_LANDAU, S, GA>(theta, a, s);
    case GF_COULOMB: return launch_theta<R, GF_COULOMB, S, GA>(theta, a, s);
    case GF_MAG: return launch_theta<R, GF_MAG, S, GA>(theta, a, s);
    default: return launch_theta<R, GF_U1XU1, S, GA>(theta, a, s);
    }
}

template <>
hipError_t launch_sweep<double>(int stride, int gauge, int theta, bool gacc, const SweepArgs<double> &a, hipStream_t s)
{
    if (gacc) return hipErrorInvalidValue;  // the FP64 phase works on the transformed links directly
    if (stride == kTiled12) return launch_g<double, kTiled12, false>(gauge, theta, a, s);
    if (stride == 18) return launch_g<double, 18, false>(gauge, theta, a, s);
    return launch_g<double, 12, false>(gauge, theta, a, s);
}

template <>
hipError_t launch_sweep<float>(int stride, int gauge, int theta, bool gacc, const SweepArgs<float> &a, hipStream_t s)
{
    if (stride != 12) return hipErrorInvalidValue;  // FP32 works on the compact layout
    if (gacc) return launch_g<float, 12, true>(gauge, theta, a, s);
    return launch_g<float, 12, false>(gauge, theta, a, s);
}

}  // namespace fast
}  // namespace su3gf
