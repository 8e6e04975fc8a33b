"""Link sweeps and projectSU3 on configurations beyond the 256 MB Infinity
Cache, whose kernels stream part of the links past the caches: bit for bit the
oracle's, on ragged extents, with the boundary between kept and streamed links
inside a direction and (half a parity's sites not being whole tiles of 64)
inside a tile."""
import ctypes as C

import numpy as np
import pytest

from oracle_lib import LANDAU, MAG, MICRO, OR

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
