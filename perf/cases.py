"""The work a gauge-fixing program has this library do, as cases to measure.

A case is a dict of plain values; ``prepare`` makes the configuration a
program holds before the call, ``run`` is one pass through the public entry
points and returns what the program would keep, ``work`` the bytes and
operations that pass cannot do without, and ``exact`` the same pass in plain
torch, in 64 bits.  ``kind`` says which entry points a case goes through:

* ``or``: the reference apps' overrelaxation loop on the operator classes --
  ``sweeps`` times orStep on both parities (on a timeslice for Coulomb), then
  one quality check (GaugeFixingStats).
* ``anneal``: one temperature of the apps' annealing loop on the operator
  classes -- saStep on both parities, then three microcanonical sweeps.
* ``start``: what the apps do to a fresh gauge copy -- a random gauge
  transformation, projectSU3, the first quality check.
* ``fix``: a whole run_mixed call, to convergence or for a fixed number of
  sweeps (mode "mixed" the default 24-bit FP32 phase, "fp64" all FP64).
* ``sa``: a whole run_sa call on the gauge transformation.
* ``copies``: gauge copies of a small lattice through the batch calls,
  annealed (one launch per half-sweep) and then fixed.
"""
import math

import numpy as np
import torch

import su3_ma_gauge_gpu_amd as gf

GAUGES = {"landau": gf.LANDAU, "coulomb": gf.COULOMB, "mag": gf.MAG, "u1xu1": gf.U1XU1}
KERNELS = {
    "landau": gf.LandauKernelsSU3,
    "coulomb": gf.CoulombKernelsSU3,
    "mag": gf.MAGKernelsSU3,
    "u1xu1": gf.U1xU1KernelsSU3,
}
OMEGA = 1.7
MICRO = 3  # microcanonical sweeps per heatbath sweep, the apps' default
# annealing temperatures in the middle of each gauge's schedule
TEMPERATURE = {"landau": 0.3, "coulomb": 0.3, "mag": 0.8, "u1xu1": 2.4}


def _case(kind, gauge, dims, **more):
    c = {"kind": kind, "gauge": gauge, "nt": dims[0], "nx": dims[1], "ny": dims[2], "nz": dims[3], "dtype": "f64"}
    c.update(more)
    return c


def listed():
    return [
        # the app loop with a check after every sweep on the smallest lattice
        # of the tests and of the built applications: latency and launches
        _case("or", "landau", (8, 8, 8, 8), name="or-check-landau-8^4-f64", sweeps=1),
        # the app loop between two checks, at the size of the headline benchmark
        _case("or", "landau", (32, 32, 32, 32), name="or-landau-32^4-f64", sweeps=4),
        # the same loop of a single-precision build on a ragged lattice, MAG
        _case("or", "mag", (20, 14, 18, 22), name="or-mag-20x14x18x22-f32", dtype="f32", sweeps=4),
        # annealing with the operator classes: the largest part of an
        # application's run (1000 temperatures by default)
        _case("anneal", "landau", (32, 32, 32, 32), name="anneal-landau-32^4-f64", temperature=0.3),
        # annealing of a single-precision build, MAG, in its critical window
        _case("anneal", "mag", (24, 24, 24, 24), name="anneal-mag-24^4-f32", dtype="f32", temperature=0.8),
        # Coulomb, as the application runs it: one timeslice at a time
        _case("anneal", "coulomb", (1, 32, 32, 32), name="anneal-coulomb-slice-32^3-f64", temperature=0.3),
        # the start of a gauge copy
        _case("start", "landau", (24, 24, 24, 24), name="start-landau-24^4-f64"),
        # a small configuration fixed to the end: launch-bound throughout
        _case("fix", "landau", (12, 12, 12, 12), name="fix-landau-12^4", mode="mixed", switch=1e-6, sweeps=0),
        # the headline benchmark: 32^4 Landau to theta < 1e-12
        _case("fix", "landau", (32, 32, 32, 32), name="fix-landau-32^4", mode="mixed", switch=1e-12, sweeps=0),
        # MAG spends most of its tens of thousands of sweeps in FP64: a
        # stretch of them
        _case("fix", "mag", (24, 24, 24, 24), name="fix-mag-24^4-fp64", mode="fp64", switch=1e-6, sweeps=300),
        # a stretch of an all-FP64 run on a configuration that streams from HBM
        _case("fix", "landau", (48, 48, 48, 48), name="fix-landau-48^4-fp64", mode="fp64", switch=1e-6, sweeps=40),
        # gauge copies of a small lattice: annealing and fixing through the
        # batch calls
        _case("copies", "landau", (8, 8, 8, 8), name="copies-8-landau-8^4", copies=8, steps=100),
    ]


def _even(rng, lo, hi):
    """An even extent, spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, 2 * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 2)))


def _dims(rng, lo, hi):
    """A lattice of extents about L, each its own: most real ones are not cubes."""
    L = _even(rng, lo, hi)
    if rng.random() < 0.4:
        return (L, L, L, L)
    return tuple(_even(rng, max(lo, (2 * L) // 3), min(hi, L + L // 3)) for _ in range(4))


def draw(rng):
    kind = rng.choice(["or", "or", "anneal", "anneal", "anneal", "start", "fix", "fix", "fix", "sa", "copies"])
    dtype = rng.choice(["f64", "f64", "f32", "f32dp"])
    if kind in ("or", "anneal"):
        gauge = rng.choice(["landau", "landau", "mag", "coulomb", "u1xu1"])
        dims = _dims(rng, 6, 36)
        if gauge == "coulomb":
            dims = (1,) + dims[1:]
        if kind == "or":
            return _case(kind, gauge, dims, dtype=dtype, sweeps=rng.choice([1, 1, 4, 10]))
        t = TEMPERATURE[gauge] * rng.uniform(0.8, 1.15)
        return _case(kind, gauge, dims, dtype=dtype, temperature=round(t, 3))
    if kind == "start":
        return _case(kind, rng.choice(["landau", "mag", "u1xu1"]), _dims(rng, 6, 40), dtype=rng.choice(["f64", "f32"]))
    if kind == "fix":
        what = rng.choice(["mixed", "mixed", "fp64"])
        if what == "mixed":  # Landau and Coulomb to the end
            gauge = rng.choice(["landau", "landau", "coulomb"])
            return _case(kind, gauge, _dims(rng, 6, 24), mode="mixed", switch=rng.choice([1e-6, 1e-12]), sweeps=0)
        gauge = rng.choice(["landau", "mag", "mag", "coulomb", "u1xu1"])
        dims = _dims(rng, 8, 40)
        V = math.prod(dims)
        return _case(kind, gauge, dims, mode="fp64", switch=1e-6, sweeps=max(20, min(300, 100_000_000 // V)))
    if kind == "sa":
        return _case(kind, "landau", _dims(rng, 8, 32), steps=rng.randrange(20, 60))
    L = rng.choice([6, 8, 10, 12])
    return _case("copies", "landau", (L, L, L, L), copies=rng.randrange(4, 9), steps=rng.randrange(50, 101))


# ------------------------------------------------------------------ inputs
def _dims_of(case):
    return (case["nt"], case["nx"], case["ny"], case["nz"])


def _volume(case):
    return math.prod(_dims_of(case))


def _sites_of(dims, device):
    """Parity-split index of each site in lexicographic order, and its parity."""
    c = torch.zeros(dims, dtype=torch.int64, device=device)
    for d, n in enumerate(dims):
        shape = [1, 1, 1, 1]
        shape[d] = n
        c = c + torch.arange(n, device=device).reshape(shape)
    par = (c % 2).reshape(-1)
    V = par.numel()
    return torch.arange(V, device=device) // 2 + par * (V // 2), par.bool()


def _third_row(u):
    """Row 2 of the SU(3) matrices u (rows 0, 1 given), complex (3, 3, ...)."""
    a, b = u[0], u[1]
    cross = torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]])
    return cross.conj()


def _orthonormal(r0, r1):
    """SU(3) matrices (3, 3, n) from two rows of three complex numbers each."""
    r0 = r0 / r0.abs().square().sum(0).sqrt()
    r1 = r1 - r0 * (r1 * r0.conj()).sum(0)
    r1 = r1 / r1.abs().square().sum(0).sqrt()
    u = torch.stack([r0, r1])
    return torch.cat([u, _third_row(u)[None]])


def _links(case, seed, direction, haar):
    """The links of one direction, complex (3, 3, V) in lexicographic order:
    exp(i sum_a c_a lambda_a / 2) to second order, c_a ~ N(0, 0.25^2) as in
    the benchmark's configurations, then the gauge transformation `haar`."""
    dims, V, dev = _dims_of(case), _volume(case), torch.device("cuda")
    gen = torch.Generator(dev)
    gen.manual_seed(seed * 1000 + direction)
    c = torch.randn(8, V, dtype=torch.float64, device=dev, generator=gen) * 0.25
    h = torch.zeros(3, 3, V, dtype=torch.complex128, device=dev)
    s3 = 1 / math.sqrt(3)
    for i, v in enumerate([c[2] + c[7] * s3, -c[2] + c[7] * s3, -2 * c[7] * s3]):
        h[i, i] = v / 2
    for (i, j), (a, b) in {(0, 1): (0, 1), (0, 2): (3, 4), (1, 2): (5, 6)}.items():
        h[i, j] = torch.complex(c[a], -c[b]) / 2
        h[j, i] = h[i, j].conj()
    rows = []
    for i in range(2):
        h2 = sum(h[i, k] * h[k] for k in range(3))
        r = 1j * h[i] - h2 / 2
        r[i] += 1
        rows.append(r)
    u = _orthonormal(*rows)
    del c, h, rows
    up = torch.roll(haar.reshape((3, 3) + dims), -1, dims=2 + direction).reshape(3, 3, V)
    out = torch.empty_like(u)
    for i in range(3):
        t = sum(haar[i, k] * u[k] for k in range(3))
        for j in range(3):
            out[i, j] = sum(t[k] * up[j, k].conj() for k in range(3))
    return out


def _configuration(case, seed):
    """The 18-real parity-split array, (4, 3, 3, 2, V) reals, on the GPU."""
    dims, V, dev = _dims_of(case), _volume(case), torch.device("cuda")
    gen = torch.Generator(dev)
    gen.manual_seed(seed * 1000 + 7)
    r = torch.randn(2, 2, 3, V, dtype=torch.float64, device=dev, generator=gen)
    haar = _orthonormal(torch.complex(r[0, 0], r[0, 1]), torch.complex(r[1, 0], r[1, 1]))
    real = torch.float64 if case["dtype"] == "f64" else torch.float32
    out = torch.empty(4, 3, 3, 2, V, dtype=real, device=dev)
    idx, _ = _sites_of(dims, dev)
    for mu in range(4):
        u = _links(case, seed, mu, haar)
        out[mu, :, :, 0, idx] = u.real.to(real)
        out[mu, :, :, 1, idx] = u.imag.to(real)
    return out


def _sites_per_block(V):
    return next(n for n in (32, 16, 8, 4, 2, 1) if (V // 2) % n == 0)


def prepare(case, seed):
    kind, gauge = case["kind"], case["gauge"]
    lat = gf.Lattice(_dims_of(case), gf.F64 if case["dtype"] == "f64" else gf.F32)
    s = {"case": case, "lat": lat, "seed": seed % 1000 + 1, "counter": 0}
    if kind == "copies":
        s["src"] = [_configuration(case, 10 * seed + k) for k in range(case["copies"])]
        s["U"] = [torch.empty_like(u) for u in s["src"]]
        return s
    s["U"] = _configuration(case, seed)
    if kind in ("fix", "sa", "start"):
        s["src"] = s["U"].clone()
    if kind in ("or", "anneal", "start"):
        s["kernels"] = KERNELS[gauge](lat, dp_updates=case["dtype"] == "f32dp")
        s["stats"] = gf.GaugeFixingStats(KERNELS[gauge], s["U"].data_ptr(), lat)
        s["common"] = gf.CommonKernelsSU3(lat)
    if gauge == "coulomb" and kind in ("or", "anneal"):
        s["Udw"] = _configuration(case, seed + 500_000)
    return s


# --------------------------------------------------------------- one pass
def _check(s):
    s["stats"].generateGaugeQuality()
    return s["stats"].getCurrentGff(), s["stats"].getCurrentA()


def run(s):
    case, lat, U = s["case"], s["lat"], s["U"]
    kind, gauge = case["kind"], GAUGES[case["gauge"]]
    if kind in ("or", "anneal", "start"):
        k, nsb = s["kernels"], _sites_per_block(lat.V)
        launch = (lat.V // 2 // nsb, 8 * nsb)
        links = (U.data_ptr(), s["Udw"].data_ptr()) if "Udw" in s else (U.data_ptr(),)
        out = {"U": U}
        if "Udw" in s:
            out["Udw"] = s["Udw"]
    if kind == "or":
        for _ in range(case["sweeps"]):
            k.orStep(*launch, *links, None, 0, OMEGA)
            k.orStep(*launch, *links, None, 1, OMEGA)
        out["gff"], out["theta"] = _check(s)
        return out
    if kind == "anneal":
        for parity in (0, 1):
            k.saStep(*launch, *links, None, parity, case["temperature"], s["seed"], s["counter"])
            s["counter"] += 1
        for _ in range(MICRO):
            k.microStep(*launch, *links, None, 0)
            k.microStep(*launch, *links, None, 1)
        return out
    if kind == "start":
        U.copy_(s["src"])
        for parity in (0, 1):
            k.randomTrafo(*launch, *links, None, parity, s["seed"], s["counter"])
            s["counter"] += 1
        s["common"].projectSU3(lat.V // nsb, nsb, U.data_ptr())
        out["gff"], out["theta"] = _check(s)
        return out
    if kind == "fix":
        U.copy_(s["src"])
        more = {}
        if case["sweeps"]:  # a stretch of a longer run: the precision is not met
            more = {"maxiter": case["sweeps"]}
        r = gf.run_mixed(lat, U.data_ptr(), gauge, OMEGA, case["switch"], 1e-12,
                         mode=gf.MIXED_FP64 if case["mode"] == "fp64" else gf.MIXED_GAUGE24, **more)
        return {"U": U, "gff": r.gff, "theta": r.theta, "sweeps": r.sweeps}
    if kind == "sa":
        U.copy_(s["src"])
        counter, ntemps = gf.run_sa(lat, U.data_ptr(), gauge, 0.4, 0.01, case["steps"], MICRO, seed=s["seed"], mode=2)
        return {"U": U, "counter": counter, "temperatures": ntemps}
    # copies: the copies' links are in place before the batch's streams use them
    n = case["copies"]
    for u, src in zip(U, s["src"]):
        u.copy_(src)
    gf.synchronize()
    ptrs = [u.data_ptr() for u in U]
    gf.batch_run_sa([lat] * n, ptrs, gauge, 1.45, 0.01, case["steps"], MICRO, seeds=[s["seed"]] * n,
                    counters=[100_000 * c for c in range(n)], mode=2, one_launch=True)
    res = gf.batch_run_mixed([lat] * n, ptrs, gauge, OMEGA, 1e-12, 1e-12)
    return {"U": list(U), "gff": [r.gff for r in res], "sweeps": [r.sweeps for r in res]}


# -------------------------------------------------------- bytes, operations
FLOPS_SITE = 2252 + 22  # one site's update, as the reference apps count it


def work(case):
    """Per half-sweep on the links: rows 0, 1 of each link once in and once
    out.  Per half-sweep of a run on the gauge transformation: each link read
    once in the form it is held in (36 B a link in 24 bits, 96 B in FP64),
    each site's transformation (rows 0, 1) once in and half of them once out."""
    V = _volume(case)
    real = 8 if case["dtype"] == "f64" else 4
    links = 4 * V * 12 * real  # rows 0, 1 of the configuration
    kind = case["kind"]
    coulomb = case["gauge"] == "coulomb"
    # a timeslice's sweep touches the time links of the slice and the one before
    touched = links * 5 // 4 if coulomb and kind in ("or", "anneal") else links
    if kind == "or":
        n = 2 * case["sweeps"]
        return {"bytes": n * 2 * touched + links, "flops": n / 2 * V * FLOPS_SITE}
    if kind == "anneal":
        n = 2 * (1 + MICRO)
        return {"bytes": n * 2 * touched, "flops": n / 2 * V * FLOPS_SITE}
    if kind == "start":
        whole = 4 * V * 18 * real
        return {"bytes": 2 * whole + 2 * 2 * links + links + whole + links, "flops": 2 * V * FLOPS_SITE}
    copies = case.get("copies", 1)
    form = 96 if case.get("mode") == "fp64" else 36
    g = 96 if case.get("mode") == "fp64" else 48
    half = 4 * V * form + V * g + V // 2 * g
    if kind == "fix":
        # about 3 L^2 sweeps to convergence with overrelaxation
        sweeps = case["sweeps"] or 3 * max(_dims_of(case)) ** 2
    else:
        sweeps = case["steps"] * (1 + MICRO) + (3 * max(_dims_of(case)) ** 2 if kind == "copies" else 0)
    whole = 4 * V * 18 * real
    return {"bytes": copies * (4 * whole + 2 * sweeps * half), "flops": copies * sweeps * V * FLOPS_SITE}


# ------------------------------------------------- the same pass in 64 bits
SUBGROUPS = ((0, 2), (1, 2), (0, 1))


class _Links:
    """A configuration as complex128 (4, 3, 3, Nt, Nx, Ny, Nz), rows 0, 1 of
    the stored links and the third rebuilt; down[mu] = U_mu(x - mu)."""

    def __init__(self, U, dims, Udw=None):
        self.dims = dims
        self.idx, odd = _sites_of(dims, U.device)
        self.odd = odd.reshape(dims)
        self.u = self._read(U)
        self.dw = self._read(Udw)[0] if Udw is not None else None  # the time links of slice t - 1

    def _read(self, U):
        u = torch.complex(U[:, :, :, 0].double(), U[:, :, :, 1].double())[..., self.idx]
        for mu in range(4):
            row = _third_row(u[mu])
            u[mu, 2] = row / row.abs().square().sum(0).sqrt()
        return u.reshape((4, 3, 3) + self.dims)

    def down(self, mu):
        if mu == 0 and self.dw is not None:
            return self.dw
        return torch.roll(self.u[mu], 1, dims=2 + mu)

    def put_down(self, mu, v):
        if mu == 0 and self.dw is not None:
            self.dw = v
        else:
            self.u[mu] = torch.roll(v, -1, dims=2 + mu)

    def write(self, like):
        """(4, 3, 3, 2, V) reals: rows 0, 1, and the third as stored in like."""
        out = like.double().clone()
        u = self.u.reshape(4, 3, 3, -1)
        for i in range(2):
            out[:, i, :, 0][..., self.idx] = u[:, i].real
            out[:, i, :, 1][..., self.idx] = u[:, i].imag
        return out


def _quaternion(gauge, U, i, j, omega):
    """The overrelaxed SU(2) element (q0..q3) of every site and subgroup (i, j)."""
    s = [0, 0, 0, 0]
    for mu in range(4):
        if gauge == "coulomb" and mu == 0:
            continue
        for up, m in ((True, U.u[mu]), (False, U.down(mu))):
            a00, a01, a10, a11 = m[i, i], m[i, j], m[j, i], m[j, j]
            if gauge == "mag":
                d = a00.abs().square() - a01.abs().square() - a10.abs().square() + a11.abs().square()
                c = a00 * a10.conj() - a01 * a11.conj() if up else a00.conj() * a01 - a10.conj() * a11
                q = (d, c.imag, c.real, torch.zeros_like(d))
            else:
                f = -1 if up else 1
                q = (a00.real + a11.real, f * (a01.imag + a10.imag), f * (a01.real - a10.real),
                     f * (a00.imag - a11.imag))
            s = [x + y for x, y in zip(s, q)]
    if gauge == "mag":
        s[1], s[2] = 2 * s[1], 2 * s[2]
        s[0] = s[0] + (s[0] ** 2 + s[1] ** 2 + s[2] ** 2).sqrt()
    elif gauge == "u1xu1":
        s[1], s[2] = torch.zeros_like(s[1]), torch.zeros_like(s[2])
    ai, a0 = s[1] ** 2 + s[2] ** 2 + s[3] ** 2, s[0] ** 2
    b = (omega * a0 + ai) / (a0 + ai)
    c = 1 / (a0 + b * b * ai).sqrt()
    return s[0] * c, s[1] * b * c, s[2] * b * c, s[3] * b * c


def _half_sweep(gauge, U, parity, omega):
    here = U.odd if parity else ~U.odd
    for i, j in SUBGROUPS:
        q = _quaternion(gauge, U, i, j, omega)
        q = [torch.where(here, v, torch.full_like(v, 1.0 if k == 0 else 0.0)) for k, v in enumerate(q)]
        g00, g01 = torch.complex(q[0], q[3]), torch.complex(q[2], q[1])
        for mu in range(4):
            m = U.u[mu]
            a, b = m[i].clone(), m[j].clone()
            m[i], m[j] = g00 * a + g01 * b, g00.conj() * b - g01.conj() * a
            d = U.down(mu).clone()
            a, b = d[:, i].clone(), d[:, j].clone()
            d[:, i], d[:, j] = a * g00.conj() + b * g01.conj(), b * g00 - a * g01
            U.put_down(mu, d)


def _quality(gauge, U):
    """(gff, theta) with the reference's prefactors."""
    V = math.prod(U.dims)
    mus = [mu for mu in range(4) if not (gauge == "coulomb" and mu == 0)]
    if gauge == "mag":
        g = sum(float(U.u[mu, j, j].abs().square().sum()) for mu in mus for j in range(3))
        th = 0.0
        for i, j in ((0, 1), (0, 2), (1, 2)):
            x = 0
            for mu in mus:
                a, d = U.u[mu], U.down(mu)
                x = x + a[i, i] * a[j, i].conj() - a[i, j] * a[j, j].conj()
                x = x + d[i, i].conj() * d[i, j] - d[j, i].conj() * d[j, j]
            th += float(x.abs().sum())
    else:
        g = sum(float(U.u[mu, j, j].real.sum()) for mu in mus for j in range(3))
        s = sum(U.u[mu] - U.down(mu) for mu in mus)
        tr = (s[0, 0] + s[1, 1] + s[2, 2]) / 3
        for i in range(3):
            s[i, i] = s[i, i] - tr
        th = sum(float((s[i, j] - s[j, i].conj()).abs().square().sum()) for i in range(3) for j in range(3))
    return g / (9 if gauge == "coulomb" else 12) / V, th / 3 / V


def exact(case, seed):
    """Overrelaxation loops, and all-FP64 runs of a fixed number of sweeps, in
    plain torch.  (A heatbath's accept-or-reject steps and a run's stopping
    sweep follow the rounding of the precision they run in; the FP32 phase of
    a mixed run is not a 64-bit computation.)"""
    kind, gauge, V = case["kind"], case["gauge"], _volume(case)
    if kind == "or":
        n = case["sweeps"]
    elif kind == "fix" and case["mode"] == "fp64" and case["sweeps"] * V < 250_000_000:
        n = case["sweeps"]
    else:
        return None
    start = _configuration(case, seed)
    slice_ = gauge == "coulomb" and kind == "or"
    dw = _configuration(case, seed + 500_000) if slice_ else None
    U = _Links(start, _dims_of(case), dw)
    omega = float(np.float32(OMEGA))
    for _ in range(n):
        _half_sweep(gauge, U, 0, omega)
        _half_sweep(gauge, U, 1, omega)
    gff, theta = _quality(gauge, U)
    if kind == "fix":
        full = torch.empty(start.shape, dtype=torch.float64, device=start.device)
        flat = U.u.reshape(4, 3, 3, -1)
        full[:, :, :, 0][..., U.idx] = flat.real
        full[:, :, :, 1][..., U.idx] = flat.imag
        # a Coulomb run reports its worst timeslice's theta
        return {"U": full, "gff": gff, "theta": None if gauge == "coulomb" else theta, "sweeps": None}
    out = {"U": U.write(start), "gff": gff, "theta": theta}
    if slice_:
        v = dw.double().clone()
        w = U.dw.reshape(3, 3, -1)
        for i in range(2):
            v[0, i, :, 0][..., U.idx] = w[i].real
            v[0, i, :, 1][..., U.idx] = w[i].imag
        out["Udw"] = v
    return out
