"""Heatbath steps at temperatures where most attempts are rejected, so that a
wave's lanes make the attempts of the sites left together (and, at a few
hundred attempts per site, draw some uniforms again): the oracle's links,
which makes them one after another.  As for every heatbath step (log, cospi and
sinpi are the device's and the host's), to 1e-10."""
import numpy as np
import pytest

from oracle_lib import LANDAU, MAG, SA, U1XU1, rows01

pytestmark = pytest.mark.gpu
KERNELS = {LANDAU: "LandauKernelsSU3", MAG: "MAGKernelsSU3", U1XU1: "U1xU1KernelsSU3"}


def _hot(oracle, dims, counter):
    U = np.empty(72 * int(np.prod(dims)), oracle.np_real)
    oracle.set_hot(dims, U, 11, counter)
    return U


# whole waves, a partial last wave, less than one wave
@pytest.mark.parametrize("dims", [(4, 4, 4, 8), (6, 6, 6, 6), (2, 2, 4, 4)])
@pytest.mark.parametrize("gauge,T", [(LANDAU, 0.4), (LANDAU, 60.0), (MAG, 0.8), (MAG, 100.0), (U1XU1, 2.4), (U1XU1, 30.0)])
def test_rejected_attempts(gf, gpu, oracle, gauge, T, dims):
    V = int(np.prod(dims))
    lat = gf.Lattice(dims)
    U = _hot(oracle, dims, 1)
    d = gf.DeviceBuffer.from_numpy(U)
    K = getattr(gf, KERNELS[gauge])(lat)
    for parity in (0, 1):
        print("heatbath", gauge, T, dims, parity, flush=True)
        K.saStep(V // 2, 8, d, None, parity, T, 7, 3 + parity)
        oracle.sweep(gauge, SA, dims, U, parity, T, 7, 3 + parity, nsb=1)
    assert np.abs(rows01(d.download(np.float64), V) - rows01(U, V)).max() < 1e-10


def test_rejected_attempts_dp_update(gf, gpu, oracle32dp):
    """FP32 links with the heatbath in double (float uniforms): to float rounding."""
    dims = (6, 6, 6, 6)
    V = int(np.prod(dims))
    U = _hot(oracle32dp, dims, 2)
    lat = gf.Lattice(dims, gf.F32)
    d = gf.DeviceBuffer.from_numpy(U)
    K = gf.U1xU1KernelsSU3(lat, dp_updates=True)
    for parity in (0, 1):
        K.saStep(V // 2, 8, d, None, parity, 30.0, 7, 5 + parity)
        oracle32dp.sweep(U1XU1, SA, dims, U, parity, 30.0, 7, 5 + parity, nsb=1)
    assert np.abs(rows01(d.download(np.float32), V) - rows01(U, V)).max() < 2e-5


def test_rejected_attempts_coulomb_slice(gf, gpu, oracle):
    dims = (1, 6, 6, 6)
    V = int(np.prod(dims))
    up, dw = _hot(oracle, dims, 3), _hot(oracle, dims, 4)
    du, dd = gf.DeviceBuffer.from_numpy(up), gf.DeviceBuffer.from_numpy(dw)
    K = gf.CoulombKernelsSU3(gf.Lattice(dims))
    for parity in (0, 1):
        K.saStep(V // 2, 8, du, dd, None, parity, 40.0, 7, 9 + parity)
        oracle.sweep_coulomb(SA, dims, up, dw, parity, 40.0, 7, 9 + parity, nsb=1)
    assert np.abs(rows01(du.download(np.float64), V) - rows01(up, V)).max() < 1e-10
    assert np.abs(rows01(dd.download(np.float64), V) - rows01(dw, V)).max() < 1e-10
