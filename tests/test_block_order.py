"""The order in which a launch's blocks walk a lattice
(su3_ma_gauge_gpu_amd/csrc/su3gf_order.h), on the CPU: for every count of
blocks and timeslices up to a few hundred, the shapes of real lattices and
every span, each logical block runs exactly once and the rest of the grid is
padding; and where each XCD has whole timeslices of its own, it gets exactly
those, t innermost."""
import shutil
import subprocess
from pathlib import Path

import pytest

HEADER = Path(__file__).resolve().parent.parent / "su3_ma_gauge_gpu_amd" / "csrc" / "su3gf_order.h"

CHECK = r"""
#include <cstdio>
#include <vector>
#include "su3gf_order.h"
using namespace su3gf;
static int check(int64_t n, int Nt, int request)
{
    const BlockOrder o = make_block_order(n, Nt, request);
    std::vector<char> seen(n, 0);
    int64_t runs = 0;
    for (int64_t b = 0; b < order_grid(o); b++) {
        const int64_t L = ordered_block(o, (uint32_t)b);
        if (L < 0) continue;
        if (L >= n || seen[L]) { printf("n %lld Nt %d request %d: block %lld -> %lld\n", (long long)n, Nt, request, (long long)b, (long long)L); return 1; }
        seen[L] = 1;
        runs++;
    }
    if (runs != n) { printf("n %lld Nt %d request %d: %lld of them run\n", (long long)n, Nt, request, (long long)runs); return 1; }
    if (order_grid(o) > n + Nt + 8) { printf("n %lld Nt %d: grid %lld\n", (long long)n, Nt, (long long)order_grid(o)); return 1; }
    if (Nt % 8 == 0 && n % Nt == 0) {  // whole timeslices, Nt / 8 per XCD, in passes of the span
        const int64_t Q = n / Nt, own = Nt / 8;
        for (int64_t b = 0; b < n; b++) {
            const int64_t x = b % 8, k = b / 8, P = o.span, pass = k / (P * Q), r = k % (P * Q);
            if (ordered_block(o, (uint32_t)b) != (x * own + pass * P + r % P) * Q + r / P) { printf("n %lld Nt %d: place of %lld\n", (long long)n, Nt, (long long)b); return 1; }
        }
    }
    return 0;
}
int main()
{
    int bad = 0;
    for (int Nt = 1; Nt <= 24; Nt++)
        for (int64_t n = 1; n <= 300; n++)
            for (int request : {0, 1, 2, 3, 5, 11}) bad |= check(n, Nt, request);
    for (int L = 4; L <= 80; L += 2) {
        const int64_t V = (int64_t)L * L * L * L;
        for (int request = 0; request <= 18; request++) bad |= check((V / 2 + 63) / 64, L, request);  // sweeps
        bad |= check((V / 2 + 127) / 128, L, 0);  // the quality kernel
        bad |= check((int64_t)L * ((V / L / 2 + 63) / 64), L, 0);  // Coulomb's blocks per timeslice
    }
    bad |= check((int64_t)34 * 30 * 32 * 26 / 128, 34, 17);
    return bad;
}
"""


def test_every_block_once(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(CHECK)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", f"-I{HEADER.parent}", str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout[:2000]
