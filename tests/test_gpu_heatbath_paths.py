"""The heatbath's other forms against the oracle, which makes attempts one after
another and every site's update by itself: links put aside meanwhile (more
than 512 blocks), links streamed past the caches (beyond 256 MB), plain FP32,
and the annealing of the gauge transformation.

In FP64, and with the update in double, log, cospi and sinpi of device and host
differ in the last bits: 1e-10, and float rounding (2e-5).  In FP32 a last bit
also turns an accept into a reject about once in 10^7 attempts, and U1xU1's
normalisation of (q0, q3) magnifies the rest: links perturbed by 3e-7 before a
pair of the oracle's half-sweeps leave no link of Landau off by 1e-3 and 0.6%
of U1xU1's by 1e-2.  Draws taken from a wrong place in the stream give
independent elements, off by order 1 wherever an attempt was rejected."""
import numpy as np
import pytest

from oracle_lib import LANDAU, MAG, RANDOM, SA, SR, U1XU1, rows01

pytestmark = pytest.mark.gpu
KERNELS = {LANDAU: "LandauKernelsSU3", MAG: "MAGKernelsSU3", U1XU1: "U1xU1KernelsSU3"}


def _hot(gf, dims, dtype, counter):
    """Random SU(3) links, made on the device (pinned to the oracle's elsewhere)."""
    lat = gf.Lattice(dims, dtype)
    d = gf.DeviceBuffer(lat.nbytes)
    gf.CommonKernelsSU3(lat).setHot(lat.V, 1, d, None, 3, counter)
    return lat, d, d.download(lat.np_dtype)


def _step(gf, lat, d, ora, U, gauge, algo, param, dp=False):
    K = getattr(gf, KERNELS[gauge])(lat, dp_updates=dp)
    n = lat.V // 2
    for parity in (0, 1):
        print("step", lat.dims, gauge, algo, param, parity, flush=True)
        if algo == SA:
            K.saStep(n, 8, d, None, parity, param, 7, 20 + parity)
        elif algo == SR:
            K.srStep(n, 8, d, None, parity, param, 7, 20 + parity)
        else:
            K.randomTrafo(n, 8, d, None, parity, 7, 20 + parity)
        ora.sweep(gauge, algo, lat.dims, U, parity, param, 7, 20 + parity, nsb=1)
    return np.abs(rows01(d.download(lat.np_dtype), lat.V) - rows01(U, lat.V))


def _off(diff, by):
    """The share of links off by more than `by`."""
    return (diff.max(axis=1) > by).mean()


# 512 blocks, the last size with the links in registers, and 576
@pytest.mark.parametrize("dims", [(16, 16, 16, 16), (16, 16, 18, 16)])
@pytest.mark.parametrize("gauge,algo,param", [(LANDAU, SA, 0.3), (LANDAU, SA, 60.0), (MAG, SA, 0.8), (U1XU1, SA, 2.4),
                                              (MAG, SR, 0.5)])
@pytest.mark.parametrize("kind", ["f64", "f32", "f32dp"])
def test_more_blocks_than_registers_for_them(gf, gpu, oracle, oracle32, oracle32dp, kind, gauge, algo, param, dims):
    ora = {"f64": oracle, "f32": oracle32, "f32dp": oracle32dp}[kind]
    lat, d, U = _hot(gf, dims, gf.F64 if kind == "f64" else gf.F32, 1)
    diff = _step(gf, lat, d, ora, U, gauge, algo, param, dp=kind == "f32dp" and algo == SA)
    if algo == SR:
        assert diff.max() == 0
    elif kind == "f32":
        assert _off(diff, 1e-2) < 0.01
    else:
        assert diff.max() < (1e-10 if kind == "f64" else 2e-5)


# FP64 rows 0, 1: 329 MB; FP32: 300 MB
@pytest.mark.parametrize("kind,dims", [("f64", (28, 30, 30, 34)), ("f32", (34, 36, 34, 38))])
@pytest.mark.parametrize("gauge,algo,param", [(LANDAU, SA, 0.4), (MAG, SR, 0.5), (U1XU1, RANDOM, 0.0)])
def test_streamed_links(gf, gpu, oracle, oracle32, gauge, algo, param, kind, dims):
    lat, d, U = _hot(gf, dims, gf.F64 if kind == "f64" else gf.F32, 2)
    diff = _step(gf, lat, d, oracle if kind == "f64" else oracle32, U, gauge, algo, param)
    if algo == SR:
        assert diff.max() == 0
    elif kind == "f64":
        assert diff.max() < 1e-10
    else:
        assert _off(diff, 1e-2) < 0.01


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("gauge,temps,by,share", [(LANDAU, [0.4], 1e-2, 0.01), (LANDAU, [60.0], 1e-2, 0.01),
                                                  (U1XU1, [30.0, 29.0], 0.1, 0.05)])
def test_annealing_of_the_gauge_transformation(gf, gpu, oracle32, gauge, temps, by, share, mode):
    """run_sa on FP32 and on 24-bit links, without microcanonical steps: the
    oracle's FP32 heatbath on the links (U1xU1 visits both ends of its range;
    two perturbed sweeps leave 1.3% of its links off by 1e-2)."""
    dims = (6, 6, 6, 8)
    V = int(np.prod(dims))
    _, _, U = _hot(gf, dims, gf.F32, 3)
    lat = gf.Lattice(dims)
    d = gf.DeviceBuffer.from_numpy(U.astype(np.float64))
    counter, visited = gf.run_sa(lat, d, gauge, temps[0], temps[-1] if len(temps) > 1 else 0.01, 1, 0, seed=7,
                                 counter=40, mode=mode)
    assert visited == len(temps) and counter == 40 + 2 * visited
    for k, T in enumerate(temps):
        for parity in (0, 1):
            oracle32.sweep(gauge, SA, dims, U, parity, T, 7, 40 + 2 * k + parity)
    oracle32.project_all(dims, U)
    assert _off(np.abs(rows01(d.download(np.float64), V) - rows01(U, V)), by) < share
