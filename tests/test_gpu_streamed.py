"""Sweeps and projectSU3 on configurations beyond the 256 MB Infinity Cache,
whose kernels stream part of the links past the caches: bit for bit the
oracle's (link sweeps) or the unstreamed sweep's, on ragged extents, with the
boundary between kept and streamed links inside a direction and (half a
parity's sites not being whole tiles of 64) inside a tile.  And the block
order of ragged lattices."""
import ctypes as C

import numpy as np
import pytest

from oracle_lib import COULOMB, LANDAU, MAG, MICRO, OR

pytestmark = pytest.mark.gpu


def _hot(gf, dims, dtype, counter):
    """Random SU(3) links, made on the device (the oracle's setHot is pinned elsewhere)."""
    lat = gf.Lattice(dims, dtype)
    d = gf.DeviceBuffer(lat.nbytes)
    gf.CommonKernelsSU3(lat).setHot(lat.V, 1, d, None, 3, counter)
    return lat, d


# FP64 (rows 0, 1: 329 MB), FP32 (300 MB, kept up to the third direction)
@pytest.mark.parametrize("dtype,dims", [("f64", (28, 30, 30, 34)), ("f32", (34, 36, 34, 38))])
@pytest.mark.parametrize("gauge,algo", [(LANDAU, OR), (MAG, OR), (LANDAU, MICRO)])
def test_streamed_sweeps_bit_exact(gf, gpu, oracle, oracle32, gauge, algo, dtype, dims):
    ora = oracle if dtype == "f64" else oracle32
    lat, d = _hot(gf, dims, gf.F64 if dtype == "f64" else gf.F32, 1)
    U = d.download(lat.np_dtype)
    print("streamed", dtype, dims, gauge, algo, flush=True)
    for parity in (0, 1):
        gf._lib.call("gf_sweep", C.byref(lat.struct), C.c_void_p(d.ptr), None, parity, gauge, algo, C.c_float(1.7),
                     0, C.c_uint32(0), 0, None)
        ora.sweep(gauge, algo, dims, U, parity, 1.7)
    assert np.array_equal(d.download(lat.np_dtype), U)


@pytest.mark.parametrize("dtype,dims", [("f64", (28, 30, 30, 34)), ("f64", (24, 26, 26, 28)), ("f32", (34, 36, 34, 38))])
def test_streamed_project_bit_exact(gf, gpu, oracle, oracle32, dtype, dims):
    """(24, 26, 26, 28): rows 0, 1 fit the cache, all three rows (262 MB) do not."""
    ora = oracle if dtype == "f64" else oracle32
    lat, d = _hot(gf, dims, gf.F64 if dtype == "f64" else gf.F32, 2)
    U = d.download(lat.np_dtype)
    U *= lat.np_dtype(1.001)  # off the group
    d.upload(U)
    print("streamed project", dtype, dims, flush=True)
    gf.CommonKernelsSU3(lat).projectSU3(lat.V, 1, d)
    ora.project_all(dims, U)
    assert np.array_equal(d.download(lat.np_dtype), U)


def test_streamed_coulomb_slice_bit_exact(gf, gpu, oracle):
    """A timeslice beyond the cache (280 MB), its time links in two buffers."""
    dims = (1, 90, 90, 90)
    lat, up = _hot(gf, dims, gf.F64, 3)
    _, dw = _hot(gf, dims, gf.F64, 4)
    Uu, Ud = up.download(np.float64), dw.download(np.float64)
    for parity in (0, 1):
        gf._lib.call("gf_sweep", C.byref(lat.struct), C.c_void_p(up.ptr), C.c_void_p(dw.ptr), parity, gf.COULOMB,
                     gf.OR, C.c_float(1.7), 0, C.c_uint32(0), 0, None)
        oracle.sweep_coulomb(OR, dims, Uu, Ud, parity, 1.7)
    assert np.array_equal(up.download(np.float64), Uu) and np.array_equal(dw.download(np.float64), Ud)


def _mixed(gf, lat, d, gauge, mode, maxiter):
    """The links after maxiter sweeps (the precision is never met), and theta, gff."""
    r = gf.run_mixed(lat, d, gauge, 1.7, switch_precision=1e-30, precision=1e-30, maxiter=maxiter, mode=mode, check32=5)
    return d.download(np.float64), (r.sweeps, r.checks, r.theta, r.gff)


def _setting(gf, name, value):
    prev = C.c_int()
    gf._lib.call(name, value, C.byref(prev))
    return prev.value


# links and g beyond the cache: 24-bit 271 MB, FP64 677 MB; FP64 at 44 x 40^2
# x 42: g alone 284 MB, itself streamed.  A timeslice's sites of a parity are
# whole blocks, so the wavefront applies: it keeps every link cached
@pytest.mark.parametrize("gauge,mode,dims", [
    (LANDAU, "MIXED_GAUGE24", (36, 32, 34, 36)), (COULOMB, "MIXED_GAUGE24", (40, 36, 34, 36)),
    (MAG, "MIXED_GAUGE24", (36, 32, 34, 36)), (LANDAU, "MIXED_GAUGE32", (36, 32, 34, 36)),
    (MAG, "MIXED_FP64", (36, 32, 34, 36)), (LANDAU, "MIXED_FP64", (44, 40, 40, 42))])
def test_streamed_gauge_sweep_is_bit_identical(gf, gpu, gauge, mode, dims):
    """The two-kernel gauge-transformation sweep with its links streamed
    against the wavefront's, which does not stream: the same links, bit for
    bit, after sweeps with and without a check."""
    lat, src = _hot(gf, dims, gf.F64, 5)
    got = []
    prev = _setting(gf, "gf_set_wavefront", 0), _setting(gf, "gf_set_block_order", 0)
    try:
        for slab in (0, 6):
            _setting(gf, "gf_set_wavefront", slab)
            print("streamed gauge sweep", gauge, mode, dims, "slab", slab, flush=True)
            d = gf.DeviceBuffer(lat.nbytes)
            d.copy_from(src)
            got.append(_mixed(gf, lat, d, gauge, getattr(gf, mode), 4))
            d.free()
    finally:
        _setting(gf, "gf_set_wavefront", prev[0])
        _setting(gf, "gf_set_block_order", prev[1])
    assert got[0][1] == got[1][1]
    assert np.array_equal(got[0][0], got[1][0])


@pytest.mark.parametrize("gauge", [LANDAU, COULOMB, MAG])
@pytest.mark.parametrize("dims", [(10, 6, 6, 10), (14, 4, 6, 6), (6, 10, 6, 6), (22, 4, 6, 10)])
def test_block_order_of_ragged_lattices(gf, gpu, gauge, dims):
    """Lattices whose timeslices are no multiple of 8, nor whole 64-site
    blocks: the same links, theta and functional in every block order, and
    the FP64 run's on the link sweeps (whose blocks are in plain order)."""
    U = gf.make_config(dims, 0.3, 1, 2)
    lat = gf.Lattice(dims)
    prev = _setting(gf, "gf_set_wavefront", 0), _setting(gf, "gf_set_block_order", 0)
    try:
        for mode in ("MIXED_GAUGE24", "MIXED_FP64"):
            want = None
            for span in (0, 1, 2, 7, 11):
                _setting(gf, "gf_set_block_order", span)
                got = _mixed(gf, lat, gf.DeviceBuffer.from_numpy(U), gauge, getattr(gf, mode), 13)
                want = want or got
                assert got[1] == want[1], (mode, span)
                assert np.array_equal(got[0], want[0]), (mode, span)
    finally:
        _setting(gf, "gf_set_wavefront", prev[0])
        _setting(gf, "gf_set_block_order", prev[1])
    d = gf.DeviceBuffer.from_numpy(U)
    r = gf.run_fast(lat, d, gauge, 1.7, 1e-30, 13)
    assert (want[1][2], want[1][3]) == pytest.approx((r.theta, r.gff), rel=1e-9)
    assert np.abs(want[0] - d.download(np.float64)).max() < 1e-9
