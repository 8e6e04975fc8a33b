"""The two-kernel gauge-transformation sweep on lattices whose links (and, at
44 x 40 x 40 x 42 in FP64, g itself) are streamed past the caches, against
sweeps that share none of its streaming: the operators' sweeps of the links,
and the check of the returned links."""
import ctypes as C

import numpy as np
import pytest

from oracle_lib import LANDAU, MAG

pytestmark = pytest.mark.gpu
KERNELS = {LANDAU: "LandauKernelsSU3", MAG: "MAGKernelsSU3"}
FP64 = [(LANDAU, (44, 40, 40, 42)), (LANDAU, (36, 32, 34, 36)), (MAG, (44, 40, 40, 42)), (MAG, (36, 32, 34, 36))]


@pytest.fixture
def two_kernels(gf):
    prev = {}
    for name in ("gf_set_wavefront", "gf_set_block_order"):
        p = C.c_int()
        gf._lib.call(name, 0, C.byref(p))
        prev[name] = p.value
    yield
    for name, value in prev.items():
        gf._lib.call(name, value, None)


def _hot(gf, dims, counter):
    lat = gf.Lattice(dims)
    d = gf.DeviceBuffer(lat.nbytes)
    gf.CommonKernelsSU3(lat).setHot(lat.V, 1, d, None, 3, counter)
    return lat, d


def _copy(gf, lat, src):
    d = gf.DeviceBuffer(lat.nbytes)
    d.copy_from(src)
    return d


def _quality(gf, lat, d, gauge):
    st = gf.GaugeFixingStats(getattr(gf, KERNELS[gauge]), d, lat)
    st.generateGaugeQuality()
    return st.getCurrentA(), st.getCurrentGff()


@pytest.mark.parametrize("gauge,dims", FP64)
def test_fp64_sweeps_follow_the_link_sweeps(gf, gpu, two_kernels, gauge, dims):
    """40 sweeps: 32 with the check (the phase starts with fine checks) and
    more, after the first read, mostly without.  Rounding is 1e-16 a sweep; a
    site whose sums nearly vanish (one in 10^8) magnifies it up to 10^4 times
    and the sweeps that follow a few hundred times.  A link or g read from a
    wrong place or too early is off by order 1."""
    lat, src = _hot(gf, dims, 5)
    d = _copy(gf, lat, src)
    print("streamed fp64", gauge, dims, flush=True)
    r = gf.run_mixed(lat, d, gauge, 1.7, precision=1e-30, maxiter=40, mode=gf.MIXED_FP64)
    got = d.download(np.float64)
    d.free()
    K = getattr(gf, KERNELS[gauge])(lat)
    n = lat.V // 2
    for _ in range(40):
        for parity in (0, 1):
            K.orStep(n, 8, src, None, parity, 1.7)
    gf.CommonKernelsSU3(lat).projectSU3(lat.V, 1, src)
    want = src.download(np.float64)
    assert r.sweeps == 40 and 32 <= r.checks < 40
    np.subtract(got, want, out=got)
    assert max(got.max(), -got.min()) < 1e-9


@pytest.mark.parametrize("gauge,dims", FP64)
def test_fp64_check_is_the_returned_links(gf, gpu, two_kernels, gauge, dims):
    """A run that meets its precision reports the sweep kernels' own theta and
    functional (read-only pass, even and odd kernel): those of its links."""
    lat, src = _hot(gf, dims, 6)
    d = _copy(gf, lat, src)
    t = gf.run_mixed(lat, d, gauge, 1.7, precision=1e-30, maxiter=12, mode=gf.MIXED_FP64).theta
    d.copy_from(src)
    print("streamed check", gauge, dims, t, flush=True)
    r = gf.run_mixed(lat, d, gauge, 1.7, precision=1.001 * t, maxiter=20, mode=gf.MIXED_FP64)
    assert r.converged == 1 and r.sweeps <= 12
    assert (r.theta, r.gff) == pytest.approx(_quality(gf, lat, d, gauge), rel=1e-10)


# 24-bit links and g beyond the cache; FP32
@pytest.mark.parametrize("gauge,mode,dims", [(LANDAU, "MIXED_GAUGE24", (36, 32, 34, 36)), (MAG, "MIXED_GAUGE24", (36, 32, 34, 36)),
                                             (LANDAU, "MIXED_GAUGE32", (36, 32, 34, 36)), (LANDAU, "MIXED_GAUGE64", (36, 32, 34, 36)),
                                             (MAG, "MIXED_GAUGE64", (36, 32, 34, 36))])
def test_fp32_phase_ends_where_the_fp64_sweeps_say(gf, gpu, two_kernels, gauge, mode, dims):
    """The FP32 phase, checked every 5 sweeps at first, ends at its tenth if
    the switch lies 0.1% above the FP64 sweeps' theta after ten (and below
    that after five), and not there if it lies 0.1% below: single precision,
    1e-7 a sweep, moves theta by less.  One FP64 sweep follows."""
    lat, src = _hot(gf, dims, 7)
    d = gf.DeviceBuffer(lat.nbytes)

    def run(switch, maxiter, mode):
        d.copy_from(src)
        print("streamed fp32 phase", gauge, mode, dims, switch, maxiter, flush=True)
        return gf.run_mixed(lat, d, gauge, 1.7, switch_precision=switch, precision=1e-30, maxiter=maxiter, mode=mode,
                            check32=1)

    five, ten = (run(1e-30, n, gf.MIXED_FP64).theta for n in (5, 10))
    assert five > 1.01 * ten
    above, below = (run(f * ten, 11, getattr(gf, mode)).sweeps_fp32 for f in (1.001, 0.999))
    assert (above, below) == (10, 11)
