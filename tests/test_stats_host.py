"""The host side of a gauge-quality handle, on the CPU, with a stand-in for the
HIP runtime (tests/hip_stand_in.h): what a check's kernel needs is in
place on the check's own stream."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
SRC = ROOT / "tests" / "stats_host_check.cpp"


@pytest.fixture(scope="module")
def counts(gf, tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = tmp_path_factory.mktemp("stats") / "check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", "-rdynamic", str(SRC), "-o", str(exe), "-ldl"], check=True)
    res = subprocess.run([str(exe), str(gf._lib.LIB_PATH)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
    words = res.stdout.split()
    return {k: int(v) for k, v in zip(words[::2], words[1::2])}


def test_count_is_zero_on_the_checks_own_stream(counts):
    """A 4 x 4 x 4 x 8 check is one launch that counts its blocks in a device
    word: every launch finds it 0, by a fill that its own stream has waited for."""
    assert counts["launches"] == 3 and counts["words"] == 1
    assert counts["unordered"] == 0
    assert counts["not_zero"] == 0


def test_a_check_without_a_result_reports_none(counts):
    """Where the kernel leaves no result, theta and gff are NaN: not what the
    memory held, nor the check's before it."""
    assert counts["stale"] == 0
