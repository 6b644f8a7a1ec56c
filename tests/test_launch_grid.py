"""Grids of launches with many blocks (lpm_amd/csrc/launch_grid.hpp): fewer
than 2^32 threads in x, rows within the device's 65,536, no block missing."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = shutil.which("g++") or shutil.which("c++")

SOURCE = """
#include <cstdio>
#include "launch_grid.hpp"
int main() {
  long long blocks;
  int threads;
  while (std::scanf("%lld %d", &blocks, &threads) == 2) {
    const lpm_amd::GridXY g = lpm_amd::grid_xy(blocks, threads);
    std::printf("%u %u\\n", g.x, g.y);
  }
}
"""


@pytest.mark.skipif(CXX is None, reason="no host compiler")
def test_grid_xy(tmp_path):
    src, exe = tmp_path / "grid.cpp", str(tmp_path / "grid")
    src.write_text(SOURCE)
    subprocess.run([CXX, "-std=c++17", f"-I{ROOT}/lpm_amd/csrc", str(src),
                    "-o", exe], check=True)
    cases = [(b, t) for t in (64, 128, 256, 512)
             for most in [(2 ** 32 - 1) // t // 8 * 8]
             for b in (1, 7, 1922, most - 1, most, most + 1, 2 * most,
                       2 * most + 1, 2 ** 31 // 64 * 4)]
    out = subprocess.run([exe], input="\n".join(f"{b} {t}" for b, t in cases),
                         capture_output=True, text=True, check=True).stdout
    for (b, t), line in zip(cases, out.splitlines(), strict=True):
        x, y = map(int, line.split())
        assert x * t < 2 ** 32 and 1 <= y <= 65536
        assert b <= x * y < b + x
        if b * t < 2 ** 32 - 8 * t:
            assert (x, y) == (b, 1)
        if y > 1:
            assert x % 8 == 0
