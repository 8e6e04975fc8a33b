"""What the first call on a lattice times before it runs, on the CPU with a
stand-in for the HIP runtime (tests/hip_stand_in.h)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
SRC = ROOT / "tests" / "tuner_host_check.cpp"


@pytest.fixture(scope="module")
def timings(gf, tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = tmp_path_factory.mktemp("tuner") / "check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", "-rdynamic", str(SRC), "-o", str(exe), "-ldl"], check=True)

    def run(dims):
        res = subprocess.run([str(exe), str(gf._lib.LIB_PATH), *map(str, dims)], capture_output=True, text=True,
                             timeout=60)
        assert res.returncode == 0, res.stdout + res.stderr
        words = res.stdout.split()
        return int(words[1]), int(words[3])

    return run


# Nt no multiple of 8; timeslices that are no whole number of blocks (64 sites
# of a parity in the sweeps, 128 in the check).  The FP64 sweep's other path,
# the wavefront in slabs of 2, 3, 4, 6, 8 and 12, takes whole blocks
@pytest.mark.parametrize("dims,slabs", [((6, 6, 6, 6), 0), ((12, 12, 12, 12), 0), ((20, 20, 20, 20), 0),
                                        ((36, 36, 36, 36), 0), ((16, 6, 6, 10), 0), ((32, 6, 10, 14), 0),
                                        ((18, 16, 16, 16), 6)])
def test_ragged_lattices_time_no_block_orders(timings, dims, slabs):
    """The default order alone: first sweeps, warm-up and its time."""
    assert timings(dims) == (0, 3 + slabs)


@pytest.mark.parametrize("dims,spans", [((8, 8, 8, 8), 0), ((16, 16, 16, 16), 1), ((32, 16, 16, 16), 2), ((48, 16, 16, 16), 3)])
def test_whole_timeslices_time_the_passes(timings, dims, spans):
    """Nt / 8 timeslices to an XCD: one timing of all of them in one pass, and
    one for each proper divisor (the check; the sweeps also time the
    wavefront)."""
    assert timings(dims)[0] == (spans + 1 if spans else 0)
