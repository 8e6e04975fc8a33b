// su3gf_exact.hip -- kernels of the drop-in operator API, compiled with
// -ffp-contract=off: every multiply and add rounds separately and in the
// reference's order, sums over a site's links follow the reference's ladder
// and 1/sqrt stands for rsqrt, so an FP64 half-sweep reproduces the CPU
// restatement of the reference bit for bit.
//
// Kernels: the sweep (su3gf_sweep.h, EXACT = true), projectSU3
// (CommonKernelsSU3.hxx:71-90), setHot (CommonKernelsSU3.hxx:92-130) and the
// per-site quality (LandauKernelsSU3.hxx:114-191, CoulombKernelsSU3.hxx:110-183,
// MAGKernelsSU3.hxx:116-223) with a deterministic block reduction.
#include "su3gf_sweep.h"

namespace su3gf {
namespace exact {

static inline unsigned blocks_for(int64_t threads) { return (unsigned)((threads + kBlock - 1) / kBlock); }

// ------------------------------------------------------------------- sweep
// The half-sweep with an update that draws random numbers (heatbath,
// stochastic relaxation, random transformation): k_sweep's mapping, but one
// wave of the block makes the update and hands the SU(2) element to the
// others through LDS (two barriers per subgroup, the same values).  In
// k_sweep every wave computes its sites' update from the shared sums; a
// heatbath costs more than the rest of the kernel, so that made four waves
// repeat it, and its registers on top of the links' left 2 waves per SIMD in
// FP64 (198 VGPRs).  PARK: the updating wave puts its links aside in LDS
// meanwhile, which leaves 122 VGPRs and 4 waves per SIMD.  Heatbath half-sweep, Landau
// at T = 0.3: FP64 32^4 250 -> 175 us, 24^4 95 -> 67; FP32 32^4 129 -> 92,
// with the update in double 186 -> 118; MAG at T = 0.8, FP64 32^4 313 -> 186.
// A fifth wave for the update, without links, needs no such copy but leaves
// room for fewer blocks (FP64 Landau 32^4: 263 us).
template <typename R, int G, int A, int S, bool STREAM, bool PARK>
__global__ __launch_bounds__(kBlock) void k_sweep_rng(SweepArgs<R> a)
{
    constexpr bool kSums = A != GF_RANDOM;  // the random transformation does not read the links
    constexpr int kQ = 4 * 64;              // an SU(2) element: [comp 4][lane 64]
    constexpr int kX = 8 * 4 * 64;          // the links' contributions: [link 8][comp 4][lane 64]
    __shared__ R lds[kSums ? kQ + kX + (PARK ? 36 * 64 : 0) : 3 * kQ];
    R *const lx = lds + kQ, *const park = lds + kQ + kX;
    const int mu = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    // consecutive blocks of an XCD update with different waves, so that the
    // updates of a CU's blocks are spread over its SIMDs
    const bool updates = mu == (int)((blockIdx.x >> 3) & 3);
    bool active;
    const int64_t p = block_site(a.g, blockIdx.x, lane, active);
    const int64_t site = (active ? p : 0) + (a.parity ? a.g.Vh : 0);
    int c[4], par;
    site_coords(a.g, site, c, par);
    // Coulomb: as in k_sweep
    const bool slice_dw = G == GF_COULOMB && mu == 0 && a.g.N[0] == 1;
    const int64_t nb = slice_dw ? site : backward(a.g, c, par, mu);
    const LinkRef<R> lu = link_ref(a.U, a.g.V, S, site, mu);
    const LinkRef<R> ld = link_ref(slice_dw ? a.Udw : a.U, a.g.V, S, nb, mu);
    const bool keep_up = !STREAM || kept_link(a.keep, a.g.Vh, active ? p : 0, mu);
    const bool keep_dn = !STREAM || kept_link(a.keep, a.g.Vh, nb >= a.g.Vh ? nb - a.g.Vh : nb, mu);

    Philox rng;
    philox_init(rng, rng_tid(p, a.nsb), a.seed, a.counter);
    if (!kSums && updates) {
#pragma unroll 1
        for (int sub = 0; sub < 3; sub++) {
            const R none[8][4] = {};
            R q[4];
            site_update<R, G, A, true>(none, q, a.param, rng);
#pragma unroll
            for (int k = 0; k < 4; k++) lds[sub * kQ + k * 64 + lane] = q[k];
        }
    }

    M3<R> up, dn;
    if (active) {
        if constexpr (STREAM) {
            load12(lu, up, keep_up);
            load12(ld, dn, keep_dn);
        } else {
            load12(lu, up);
            load12(ld, dn);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) { up.e[i][j] = cx((R)(i == j), (R)0); dn.e[i][j] = up.e[i][j]; }
    }
    reconstruct_e<true>(up);
    reconstruct_e<true>(dn);
    if (!kSums) __syncthreads();

    auto subgroup = [&](auto I_, auto J_, int sub) {
        constexpr int I = decltype(I_)::value, J = decltype(J_)::value;
        R q[4];
        if (kSums) {
            R vu[4], vd[4];
            link_contrib<R, G, I, J, true>(up, vu);
            link_contrib<R, G, I, J, false>(dn, vd);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                lx[((0 + mu) * 4 + k) * 64 + lane] = vu[k];
                lx[((4 + mu) * 4 + k) * 64 + lane] = vd[k];
            }
            __syncthreads();
            if (updates) {
                if constexpr (PARK) {
#pragma unroll
                    for (int k = 0; k < 9; k++) {
                        const Cx<R> u = up.e[k / 3][k % 3], d = dn.e[k / 3][k % 3];
                        R *const b = park + 4 * k * 64 + lane;
                        b[0] = u.x; b[64] = u.y; b[128] = d.x; b[192] = d.y;
                    }
                    asm volatile("" ::: "memory");  // the links' registers are free until they come back
                }
                R cc[8][4];
#pragma unroll
                for (int m = 0; m < 8; m++)
#pragma unroll
                    for (int k = 0; k < 4; k++) cc[m][k] = lx[(m * 4 + k) * 64 + lane];
                site_update<R, G, A, true>(cc, q, a.param, rng);
#pragma unroll
                for (int k = 0; k < 4; k++) lds[k * 64 + lane] = q[k];
                if constexpr (PARK) {
                    asm volatile("" ::: "memory");
#pragma unroll
                    for (int k = 0; k < 9; k++) {
                        const R *const b = park + 4 * k * 64 + lane;
                        up.e[k / 3][k % 3] = cx(b[0], b[64]);
                        dn.e[k / 3][k % 3] = cx(b[128], b[192]);
                    }
                }
            }
            // the next writes to the exchange follow this barrier, after which
            // the update has read it; the next element is written after the
            // next exchange's barrier, past every wave's reads of this one
            __syncthreads();
        }
#pragma unroll
        for (int k = 0; k < 4; k++) q[k] = lds[(kSums ? 0 : sub * kQ) + k * 64 + lane];
        left_mult<R, I, J>(up, q);
        right_mult_dag<R, I, J>(dn, q);
    };
    subgroup(std::integral_constant<int, 0>(), std::integral_constant<int, 2>(), 0);
    subgroup(std::integral_constant<int, 1>(), std::integral_constant<int, 2>(), 1);
    subgroup(std::integral_constant<int, 0>(), std::integral_constant<int, 1>(), 2);
    if (active) {
        if constexpr (STREAM) {
            store12(lu, up, keep_up);
            store12(ld, dn, keep_dn);
        } else {
            store12(lu, up);
            store12(ld, dn);
        }
    }
}

// With the links in registers a heatbath in FP64 holds 2 waves per SIMD, so up
// to two blocks per CU run at once in any case, and the copies only lengthen
// the update.  FP64 half-sweep with the links in registers and put aside, and
// with every wave making the update as in k_sweep: Coulomb timeslice 32^3 (256
// blocks) 15.6, 16.7 and 16.0 us; Landau 512 blocks 20.5, 22.0 and 24.0, 576
// 29.1, 24.2 and 32.3, 810 34.1, 27.7 and 40.4, 1250 45.1, 36.4 and 48.6.  In
// FP32 there are registers for 3 waves (MAG: 4), and the line could lie at 768
// blocks (1024): 512 blocks 13.6, 14.2 and 14.7 us, 576 16.7, 17.3 and 19.7, 810
// 22.2, 17.9 and 22.1; MAG 810 21.7 and 22.7, 1125 28.3 and 24.9.  It lies at 512
// for every type: above it FP32 gives up 4% at most, and a type of its own
// would need a line for each gauge.  Stochastic relaxation, whose update is
// short, gives up 7% (FP64 MAG 576 blocks 15.6 and 16.8 us).
constexpr unsigned kUnparkedBlocks = 512;

template <typename R, int G, int A, int S, bool STREAM> static hipError_t launch_s(const SweepArgs<R> &a, hipStream_t s)
{
    constexpr int AB = A % kDpUpdate;  // the update rule without its precision
    const dim3 grid((unsigned)sweep_grid(a.g));
    if constexpr (AB == GF_OR || AB == GF_MICRO)
        hipLaunchKernelGGL((k_sweep<R, G, A, S, true, 0, false, STREAM>), grid, dim3(kBlock), 0, s, a);
    else if constexpr (AB == GF_RANDOM)
        hipLaunchKernelGGL((k_sweep_rng<R, G, A, S, STREAM, false>), grid, dim3(kBlock), 0, s, a);
    else if (STREAM || grid.x > kUnparkedBlocks)
        hipLaunchKernelGGL((k_sweep_rng<R, G, A, S, STREAM, true>), grid, dim3(kBlock), 0, s, a);
    else if constexpr (!STREAM)
        hipLaunchKernelGGL((k_sweep_rng<R, G, A, S, STREAM, false>), grid, dim3(kBlock), 0, s, a);
    return hipGetLastError();
}

template <typename R, int G, int A, int S> static hipError_t launch_t(SweepArgs<R> a, hipStream_t s)
{
    a.keep = kept_links(a.g.Vh, 48 * (int64_t)sizeof(R) * a.g.V);
    return a.keep < 4 * a.g.Vh ? launch_s<R, G, A, S, true>(a, s) : launch_s<R, G, A, S, false>(a, s);
}

template <typename R, int G, int S>
static hipError_t launch_a(int algo, const SweepArgs<R> &a, hipStream_t s)
{
    if constexpr (sizeof(R) == 4) {  // FP32 links, update rule in double
        switch (algo) {
        case GF_OR + kDpUpdate: return launch_t<R, G, GF_OR + kDpUpdate, S>(a, s);
        case GF_MICRO + kDpUpdate: return launch_t<R, G, GF_MICRO + kDpUpdate, S>(a, s);
        case GF_SA + kDpUpdate: return launch_t<R, G, GF_SA + kDpUpdate, S>(a, s);
        default: break;
        }
    }
    switch (algo) {
    case GF_OR: return launch_t<R, G, GF_OR, S>(a, s);
    case GF_MICRO: return launch_t<R, G, GF_MICRO, S>(a, s);
    case GF_SA: return launch_t<R, G, GF_SA, S>(a, s);
    case GF_SR: return launch_t<R, G, GF_SR, S>(a, s);
    case GF_RANDOM: return launch_t<R, G, GF_RANDOM, S>(a, s);
    default: return hipErrorInvalidValue;
    }
}

template <typename R, int S>
static hipError_t launch_g(int gauge, int algo, const SweepArgs<R> &a, hipStream_t s)
{
    switch (gauge) {
    case GF_LANDAU: return launch_a<R, GF_LANDAU, S>(algo, a, s);
    case GF_COULOMB: return launch_a<R, GF_COULOMB, S>(algo, a, s);
    case GF_MAG: return launch_a<R, GF_MAG, S>(algo, a, s);
    default: return launch_a<R, GF_U1XU1, S>(algo, a, s);
    }
}

template <typename R>
hipError_t launch_sweep(int stride, int gauge, int algo, const SweepArgs<R> &a, hipStream_t s)
{
    if (stride == 18) return launch_g<R, 18>(gauge, algo, a, s);
    return launch_g<R, 12>(gauge, algo, a, s);
}
template hipError_t launch_sweep<float>(int, int, int, const SweepArgs<float> &, hipStream_t);
template hipError_t launch_sweep<double>(int, int, int, const SweepArgs<double> &, hipStream_t);

// ----------------------------------------------------------------- project
// one thread per link.  STREAM: links beyond the Infinity Cache, of which it
// leaves the same ones in the cache as the sweeps (kept_link); the third rows,
// which no sweep reads, are streamed past it.  FP64, 18 reals, 32^4: 228 us
// with every access cached, 170 us.
template <typename R, int S, bool STREAM>
__global__ __launch_bounds__(kBlock) void k_project(R *U, int64_t V, int64_t keep, const DevState *st)
{
    if (st && st->done) return;  // a driver's run has converged: the checked state stays as it is
    const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (t >= 4 * V) return;
    const int mu = (int)(t / V);
    const int64_t idx = t - (int64_t)mu * V;
    const LinkRef<R> l = link_ref(U, V, S, idx, mu);
    const bool kept = !STREAM || kept_link(keep, V / 2, idx >= V / 2 ? idx - V / 2 : idx, mu);
    M3<R> u;
    if constexpr (STREAM) load12(l, u, kept);
    else load12(l, u);
    project_e<true>(u);
    if constexpr (STREAM) store12(l, u, kept);
    else store12(l, u);
    if (S == 18) store_row2<STREAM>(l, u);
}

template <typename R, int S>
static hipError_t launch_project_s(R *U, int64_t V, hipStream_t s, const DevState *st)
{
    const dim3 grid(blocks_for(4 * V)), block(kBlock);
    const int64_t keep = kept_links(V / 2, 48 * (int64_t)sizeof(R) * V);
    // with the third rows a configuration leaves the cache sooner
    if (keep < 2 * V || 4 * (S == 18 ? 18 : 12) * (int64_t)sizeof(R) * V > kInfinityCacheBytes)
        hipLaunchKernelGGL((k_project<R, S, true>), grid, block, 0, s, U, V, keep, st);
    else
        hipLaunchKernelGGL((k_project<R, S, false>), grid, block, 0, s, U, V, keep, st);
    return hipGetLastError();
}

template <typename R> hipError_t launch_project(int stride, R *U, int64_t V, hipStream_t s, const DevState *st)
{
    if (stride == 18) return launch_project_s<R, 18>(U, V, s, st);
    if (stride == 12) return launch_project_s<R, 12>(U, V, s, st);
    if constexpr (sizeof(R) == 8)
        if (stride == kTiled12) return launch_project_s<R, kTiled12>(U, V, s, st);
    return hipErrorInvalidValue;
}
template hipError_t launch_project<float>(int, float *, int64_t, hipStream_t, const DevState *);
template hipError_t launch_project<double>(int, double *, int64_t, hipStream_t, const DevState *);

// ----------------------------------------------------------------- set hot
// per site: identity times three random SU(2) subgroup elements from the right,
// (0,1), (0,2), (1,2), each from four uniforms in (-1,1) normalised
// (Quaternion::projectSU2, Quaternion.hxx:220-228); all 18 reals written.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_set_hot(R *U, int64_t V, uint32_t seed, uint32_t counter)
{
    const int64_t site = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (site >= V) return;
    Philox rng;
    philox_init(rng, (uint32_t)site, seed, counter);
    for (int mu = 0; mu < 4; mu++) {
        M3<R> u;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) u.e[i][j] = cx((R)(i == j ? 1 : 0), (R)0);
#define SU3GF_HOT_SUB(I, J)                                                           \
        {                                                                             \
            R q[4];                                                                   \
            _Pragma("unroll") for (int k = 0; k < 4; k++) q[k] = philox_rand(rng, R(0)) * (R)2 - (R)1; \
            const R n = (R)1 / sqrt_(q[0] * q[0] + q[3] * q[3] + q[2] * q[2] + q[1] * q[1]); \
            _Pragma("unroll") for (int k = 0; k < 4; k++) q[k] *= n;                 \
            /* right multiplication by G(q) = right_mult_dag by G(q)^dagger */       \
            const R h[4] = {q[0], -q[1], -q[2], -q[3]};                               \
            right_mult_dag<R, I, J>(u, h);                                            \
        }
        SU3GF_HOT_SUB(0, 1)
        SU3GF_HOT_SUB(0, 2)
        SU3GF_HOT_SUB(1, 2)
#undef SU3GF_HOT_SUB
        const LinkRef<R> l = link_ref(U, V, 18, site, mu);
        store12(l, u);
        store_row2(l, u);
    }
}

template <typename R>
hipError_t launch_set_hot(R *U, int64_t V, uint32_t seed, uint32_t counter, hipStream_t s)
{
    hipLaunchKernelGGL((k_set_hot<R>), dim3(blocks_for(V)), dim3(kBlock), 0, s, U, V, seed, counter);
    return hipGetLastError();
}
template hipError_t launch_set_hot<float>(float *, int64_t, uint32_t, uint32_t, hipStream_t);
template hipError_t launch_set_hot<double>(double *, int64_t, uint32_t, uint32_t, hipStream_t);

// ----------------------------------------------------------------- quality
// One thread per site, in the reference's order of operations
// (LandauKernelsSU3.hxx:114-191, CoulombKernelsSU3.hxx:110-183,
// MAGKernelsSU3.hxx:116-223): the per-site values are those of the reference
// bit for bit.  A block of 256 threads takes the 128 even and the 128 odd
// sites of parity-split index [128 L, 128 L + 128), i.e. 256 consecutive
// sites of the lexicographic order, so that most down links a site reads
// (its z and y neighbours') are the up links its own block reads, and the
// blocks are dealt out to the eight XCDs in contiguous ranges, t innermost
// (su3gf_order.h), so that the x and t neighbours' links are still in that
// XCD's L2: each link comes from HBM about once.
template <typename R, int S>
__device__ __forceinline__ void load_site_link(const QualityArgs<R> &a, int64_t idx, int mu, M3<R> &u)
{
    load12(link_ref(const_cast<R *>(a.U), a.g.V, S, idx, mu), u);
    reconstruct_e<true>(u);
}

template <typename R, int G, int S, bool SMALL>
__device__ __forceinline__ void quality_site(const QualityArgs<R> &a, int64_t site, double &dA, double &dGff)
{
    int c[4], par;
    site_coords(a.g, site, c, par);
    if (G == GF_MAG) {
        double gff = 0.0;
        double Xx[3] = {0, 0, 0}, Xy[3] = {0, 0, 0};
#pragma unroll(SMALL ? 4 : 1)
        for (int mu = 0; mu < 4; mu++) {
            M3<R> up, dw;
            load_site_link<R, S>(a, site, mu, up);
            load_site_link<R, S>(a, backward(a.g, c, par, mu), mu, dw);
#pragma unroll
            for (int j = 0; j < 3; j++) gff += (double)abs2(up.e[j][j]);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = i + 1; j < 3; j++) {
                    Cx<R> cc = up.e[i][i] * conj(up.e[j][i]) - up.e[i][j] * conj(up.e[j][j]);
                    Xx[i + j - 1] += (double)cc.x;
                    Xy[i + j - 1] += (double)cc.y;
                    // getSubgroupMatrixHermitian of the down link (SU3.hxx:231-241)
                    const Cx<R> b00 = conj(dw.e[i][i]), b01 = conj(dw.e[j][i]), b10 = conj(dw.e[i][j]),
                                b11 = conj(dw.e[j][j]);
                    cc = b00 * conj(b10) - b01 * conj(b11);
                    Xx[i + j - 1] += (double)cc.x;
                    Xy[i + j - 1] += (double)cc.y;
                }
        }
        dGff = gff;
        dA = sqrt(Xx[0] * Xx[0] + Xy[0] * Xy[0]) + sqrt(Xx[1] * Xx[1] + Xy[1] * Xy[1]) +
             sqrt(Xx[2] * Xx[2] + Xy[2] * Xy[2]);
        return;
    }
    const int mu0 = (G == GF_COULOMB) ? 1 : 0;
    M3<R> sum;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) sum.e[i][j] = cx((R)0, (R)0);
    // gff: Re tr of the up links, each trace summed from 0 in the order
    // (0,0), (1,1), (2,2), directions in order -- the reference's second loop
    // over the same links (LandauKernelsSU3.hxx:176-188), formed here from
    // the first loop's loads
    double result = 0;
    // one direction's two links at a time (140 VGPRs in FP64, 3 waves per
    // SIMD); unrolled, all eight links' loads are hoisted (256 VGPRs, 1 wave)
#pragma unroll(SMALL ? 4 : 1)
    for (int mu = mu0; mu < 4; mu++) {
        M3<R> t;
        load_site_link<R, S>(a, site, mu, t);
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) sum.e[i][j] = sum.e[i][j] + t.e[i][j];
        Cx<R> tt = cx((R)0, (R)0);
        tt = tt + t.e[0][0];
        tt = tt + t.e[1][1];
        tt = tt + t.e[2][2];
        result += (double)tt.x;
        load_site_link<R, S>(a, backward(a.g, c, par, mu), mu, t);
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) sum.e[i][j] = sum.e[i][j] - t.e[i][j];
    }
    // Sum -= Sum.trace()/3 on the diagonal; Sum -= Sum^dagger
    Cx<R> tr = cx((R)0, (R)0);
    tr = tr + sum.e[0][0];
    tr = tr + sum.e[1][1];
    tr = tr + sum.e[2][2];
    tr = cx(tr.x / (R)3, tr.y / (R)3);
#pragma unroll
    for (int i = 0; i < 3; i++) sum.e[i][i] = sum.e[i][i] - tr;
    M3<R> h;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) h.e[j][i] = conj(sum.e[i][j]);
    double prec = 0;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const Cx<R> d = sum.e[i][j] - h.e[i][j];
            prec += (double)abs2(d);
        }
    dA = prec;
    dGff = result;
}


// (theta, gff) of the lattice from its n blocks' partials in a fixed order: sum
// k (k = 0..1023) takes partials k, k + 1024, ... in order, then a fixed tree.
// NT threads make them, a thread 1024 / NT of the sums.  They go to host
// memory that the device maps.  COHERENT: partials of blocks of the same
// launch, on any XCD.
template <int NT, bool COHERENT>
__device__ __forceinline__ void reduce_partials(const double *partial, int64_t n, int crit_max, QualityResult *out)
{
    __shared__ double st[NT], sg[NT];
    constexpr int kV = 1024 / NT;
    const int t = threadIdx.x;
    const auto read = [&](int64_t k) {
        if (!COHERENT) return partial[k];
        return __longlong_as_double((int64_t)__hip_atomic_load((const uint64_t *)partial + k, __ATOMIC_RELAXED,
                                                               __HIP_MEMORY_SCOPE_AGENT));
    };
    const auto join = [&](double x, double y) { return crit_max ? fmax(x, y) : x + y; };
    double T[kV], F[kV];
#pragma unroll
    for (int v = 0; v < kV; v++) T[v] = F[v] = 0;
    for (int64_t base = 0; base < n; base += 1024)
#pragma unroll
        for (int v = 0; v < kV; v++) {
            const int64_t k = base + v * NT + t;
            if (k >= n) continue;
            T[v] = join(T[v], read(2 * k));
            F[v] += read(2 * k + 1);
        }
#pragma unroll
    for (int h = kV / 2; h >= 1; h >>= 1)
#pragma unroll
        for (int v = 0; v < h; v++) {
            T[v] = join(T[v], T[v + h]);
            F[v] += F[v + h];
        }
    st[t] = T[0];
    sg[t] = F[0];
    __syncthreads();
    for (int s = NT / 2; s >= 1; s >>= 1) {
        if (t < s) {
            st[t] = join(st[t], st[t + s]);
            sg[t] += sg[t + s];
        }
        __syncthreads();
    }
    if (t == 0) {
        out->theta = st[0];
        out->gff = sg[0];
    }
}

__global__ __launch_bounds__(1024) void k_reduce_quality(const double *partial, int64_t n, int crit_max,
                                                         QualityResult *out)
{
    reduce_partials<1024, false>(partial, n, crit_max, out);
}

// SMALL: a lattice of at most one block per CU is bound by latency.  Its
// eight links are loaded at once instead of two at a time, and with a.out the
// block that finishes last reduces the partials (written and read coherently
// at device scope, the count of finished blocks after a block's partials are
// complete).  Larger lattices keep the second kernel: their blocks would
// queue at the one count (FP32 32^4: 56 -> 79 us).  A whole check, FP64, the
// result on the host: 8^4 24.1 -> 21.3 us, 16^4 25.1 -> 23.6 us; with the
// second kernel, which no longer needs a copy after it, 24^4 44.8 -> 43.0 us,
// 32^4 101.8 -> 101.3 us.
template <typename R, int G, int S, bool SMALL>
__global__ __launch_bounds__(kBlock) void k_quality(QualityArgs<R> a)
{
    const int64_t L = ordered_block(a.order, blockIdx.x);
    const int par = threadIdx.x >= kQualitySites;
    const int64_t p = L * kQualitySites + (threadIdx.x & (kQualitySites - 1));
    const bool active = L >= 0 && p < a.g.Vh;
    double th = 0, gf = 0;
    if (active) {
        const int64_t site = p + (par ? a.g.Vh : 0);
        quality_site<R, G, S, SMALL>(a, site, th, gf);
        if (a.dGff) {
            a.dGff[site] = gf;
            a.dA[site] = th;
        }
    }
    if (!a.partial || L < 0) return;  // both uniform over the block
    __shared__ double sh[2][kBlock / 64];
    double ts = th, gs = gf;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const double o = __shfl_xor(ts, off, 64);
        ts = a.crit_max ? fmax(ts, o) : ts + o;
        gs += __shfl_xor(gs, off, 64);
    }
    const int wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        sh[0][wv] = ts;
        sh[1][wv] = gs;
    }
    __syncthreads();
    __shared__ bool last;
    if (threadIdx.x == 0) {
        double T = sh[0][0], Gs = sh[1][0];
        for (int k = 1; k < kBlock / 64; k++) {
            T = a.crit_max ? fmax(T, sh[0][k]) : T + sh[0][k];
            Gs += sh[1][k];
        }
        if (SMALL && a.out) {
            uint64_t *const o = (uint64_t *)a.partial + 2 * L;
            __hip_atomic_store(o, (uint64_t)__double_as_longlong(T), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(o + 1, (uint64_t)__double_as_longlong(Gs), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the partials are complete
            last = atomicInc(a.finished, a.order.n - 1) == a.order.n - 1;  // (wraps to 0 for the next launch)
        } else {
            a.partial[2 * L] = T;
            a.partial[2 * L + 1] = Gs;
        }
    }
    if constexpr (SMALL) {
        if (!a.out) return;
        __syncthreads();
        if (!last) return;
        reduce_partials<kBlock, true>(a.partial, a.order.n, a.crit_max, a.out);
    }
}

int64_t quality_blocks(int64_t V) { return (V / 2 + kQualitySites - 1) / kQualitySites; }

template <typename R, int S>
static hipError_t launch_quality_s(int gauge, QualityArgs<R> a, hipStream_t s)
{
    static_assert(2 * kQualitySites == kBlock, "a block holds both parities' sites");
    a.order = make_block_order(quality_blocks(a.g.V), a.g.N[0], a.tpass);
    const unsigned grid = (unsigned)order_grid(a.order);
    const bool small = a.order.n <= kSmallQualityBlocks;
    const auto launch = [&](auto G_, auto SMALL_) {
        constexpr int G = decltype(G_)::value;
        hipLaunchKernelGGL((k_quality<R, G, S, decltype(SMALL_)::value>), dim3(grid), dim3(kBlock), 0, s, a);
    };
    const auto sized = [&](auto G_) {
        if (small) launch(G_, std::true_type());
        else launch(G_, std::false_type());
    };
    if (gauge == GF_COULOMB) sized(std::integral_constant<int, GF_COULOMB>());
    else if (gauge == GF_MAG) sized(std::integral_constant<int, GF_MAG>());
    else sized(std::integral_constant<int, GF_LANDAU>());
    if (a.out && !small)
        hipLaunchKernelGGL(k_reduce_quality, dim3(1), dim3(1024), 0, s, a.partial, (int64_t)a.order.n, a.crit_max, a.out);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_quality(int stride, int gauge, const QualityArgs<R> &a, hipStream_t s)
{
    if (stride == 18) return launch_quality_s<R, 18>(gauge, a, s);
    return launch_quality_s<R, 12>(gauge, a, s);
}
template hipError_t launch_quality<float>(int, int, const QualityArgs<float> &, hipStream_t);
template hipError_t launch_quality<double>(int, int, const QualityArgs<double> &, hipStream_t);

}  // namespace exact
}  // namespace su3gf
