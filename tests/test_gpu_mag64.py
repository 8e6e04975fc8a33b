"""MAG's FP64 phase (sums of outer products of the links' columns) against the
oracle's sweeps of the links: whole blocks, partial blocks, one block; runs
that end unchecked, on the even and on the odd kernel's check."""
import numpy as np
import pytest

from oracle_lib import MAG, OR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(4, 4, 4, 8), (4, 6, 4, 8), (6, 6, 6, 6), (2, 2, 4, 4), (10, 4, 6, 2)])
@pytest.mark.parametrize("sweeps,hot", [(1, True), (2, False), (17, True), (40, False)])
def test_mag_fp64_phase_follows_the_oracle(gf, gpu, oracle, dims, sweeps, hot):
    """Rounding differs (1e-16 per sweep, amplified by a few hundred over 40
    sweeps towards the maximum): links to 1e-11, theta and gff of the final
    state to 1e-11 relative."""
    V = int(np.prod(dims))
    U = gf.make_config(dims, 0.35, 1, 2)
    if hot:
        oracle.set_hot(dims, U, 5, 1)
    lat = gf.Lattice(dims)
    d = gf.DeviceBuffer.from_numpy(U)
    print("mag64", dims, sweeps, hot, flush=True)
    r = gf.run_mixed(lat, d, gf.MAG, 1.7, precision=1e-30, maxiter=sweeps, mode=gf.MIXED_FP64)
    for _ in range(sweeps):
        for parity in (0, 1):
            oracle.sweep(MAG, OR, dims, U, parity, 1.7)
    oracle.project_all(dims, U)
    assert r.sweeps == sweeps and r.converged == 0
    assert np.abs(d.download(np.float64, 72 * V) - U).max() < 1e-11
    g, t = oracle.quality(MAG, dims, U)
    assert r.gff == pytest.approx(g, rel=1e-11)
    assert r.theta == pytest.approx(t, rel=1e-10, abs=1e-13)
