"""MAG's FP64 phase turns each link by g(x) before it forms products of its
columns, and forms those of all three columns: its rounding is that of a sweep
on the links, and it takes no column from the others by unitarity."""
import numpy as np
import pytest

from oracle_lib import from_matrices, to_matrices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [1, 3])
def test_theta_floor(gf, gpu, seed):
    """Theta where it stops falling, from a random gauge.  Products of turned
    links leave it at 1.31e-15 to 1.43e-15 (60 runs on 4^4, 6^4 and 8^4);
    products formed before the turn, whose sums are of order 8 and cancel
    after it, at 1.95e-15 to 2.07e-15.  The bound is half-way in the logarithm."""
    dims = (6, 6, 6, 6)
    lat = gf.Lattice(dims)
    d = gf.DeviceBuffer.from_numpy(gf.make_config(dims, 0.35, seed, seed + 1))
    r = gf.run_mixed(lat, d, gf.MAG, 1.7, precision=1e-30, maxiter=15000, mode=gf.MIXED_FP64)
    assert r.sweeps == 15000
    assert r.theta < 1.65e-15


# ------------------------------------------- a sweep of g on links as they are
def _cross(m):
    """Row 2 of the matrices m from rows 0, 1."""
    m[..., 2, :] = np.cross(m[..., 0, :], m[..., 1, :]).conj()
    return m


def _projected(m):
    r0 = m[..., 0, :] / np.sqrt((abs(m[..., 0, :]) ** 2).sum(-1, keepdims=True))
    r1 = m[..., 1, :] - r0 * (m[..., 1, :] * r0.conj()).sum(-1, keepdims=True)
    r1 /= np.sqrt((abs(r1) ** 2).sum(-1, keepdims=True))
    return _cross(np.stack([r0, r1, r1], -2))


def _dag(m):
    return m.conj().swapaxes(-1, -2)


def _mag_sweep(U, nn, omega):
    """One overrelaxation sweep of MAG on the gauge transformation of the links
    U[mu, site], every link turned by g and by each update."""
    V = U.shape[1]
    U = _cross(U.copy())
    g = np.tile(np.eye(3, dtype=complex), (V, 1, 1))
    for x in (np.arange(V // 2), np.arange(V // 2, V)):
        gx = g[x]
        W = []  # g(x) U g(x+mu)^dagger, and (g(x-mu) U g(x)^dagger)^dagger
        for mu in range(4):
            dn, up = nn[2 * mu][x], nn[2 * mu + 1][x]
            W.append(_cross(gx @ U[mu, x] @ _dag(g[up])))
            W.append(_dag(_cross(g[dn] @ U[mu, dn] @ _dag(gx))))
        W = np.stack(W)
        for i, j in ((0, 2), (1, 2), (0, 1)):
            a, b, c, d = W[..., i, i], W[..., i, j], W[..., j, i], W[..., j, j]
            D = (abs(a) ** 2 - abs(b) ** 2 - abs(c) ** 2 + abs(d) ** 2).sum(0)
            s = 2 * (a * c.conj() - b * d.conj()).sum(0)
            s0 = D + np.sqrt(D ** 2 + abs(s) ** 2)
            f = (omega * s0 ** 2 + abs(s) ** 2) / (s0 ** 2 + abs(s) ** 2)
            n = 1 / np.sqrt(s0 ** 2 + f ** 2 * abs(s) ** 2)
            G = np.tile(np.eye(3, dtype=complex), (len(x), 1, 1))
            G[:, i, i] = G[:, j, j] = s0 * n
            G[:, i, j], G[:, j, i] = s * f * n, -(s * f * n).conj()
            W, gx = G @ W, G @ gx
        g[x] = _projected(gx)
    # applied at the end with the third rows normalised (SU3.hxx:655-664)
    U[..., 2, :] /= np.sqrt((abs(U[..., 2, :]) ** 2).sum(-1, keepdims=True))
    return np.stack([_projected(g @ U[mu] @ _dag(g[nn[2 * mu + 1]])) for mu in range(4)])


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("dims", [(4, 4, 4, 8), (6, 6, 6, 6)])
def test_first_sweep(gf, gpu, oracle, dims, single):
    """Links unitary to double and to single precision (rows 0, 1 as they are,
    the third rebuilt): the sweep above to its rounding, 1e-16 times a few
    hundred operations.  A column taken from the others by unitarity would be
    off by the links' own rounding, 1e-8 and more."""
    V = int(np.prod(dims))
    U = gf.make_config(dims, 0.35, 1, 2)
    if single:
        U = U.astype(np.float32).astype(np.float64)
    nn = oracle.neighbour_table(dims).reshape(8, V)
    want = from_matrices(_mag_sweep(to_matrices(U, V), nn, float(np.float32(1.7))))
    d = gf.DeviceBuffer.from_numpy(U)
    r = gf.run_mixed(gf.Lattice(dims), d, gf.MAG, 1.7, precision=1e-30, maxiter=1, mode=gf.MIXED_FP64)
    assert r.sweeps == 1
    assert np.abs(d.download(np.float64, 72 * V) - want).max() < 1e-12
