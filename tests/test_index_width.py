"""Element indexes of grids too large to allocate in a test, formed on the CPU
by the kernels' own functions: the host side of the march's header, compiled
for the host alone."""
import os
import subprocess

import pytest

from evora_amd import build

SRC = """
#include <cstdio>
#include <cstdlib>
#include "fused_core.h"
int main(int argc, char **argv) {
  evh::KParams P = {};
  evh::core::Geo G = {};
  P.boundtype = std::atoi(argv[1]);
  G.nx = std::atoi(argv[2]);
  G.ny = std::atoi(argv[3]);
  for (int i = 4; i + 1 < argc; i += 2) {
    const long long c = (long long)evh::core::col_offset(P, G, std::atoi(argv[i]), std::atoi(argv[i + 1]));
    std::printf("%lld\\n", c);
  }
}
"""


@pytest.mark.parametrize("nx,ny", [(1 << 16, (1 << 15) + 7), (30000, 99999), (65000, 46000), (12, 5)])
@pytest.mark.parametrize("bound", [1, 2])
def test_column_offsets_of_planes_above_2_31_cells(tmp_path, nx, ny, bound):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    exe = tmp_path / "cols"
    (tmp_path / "cols.hip").write_text(SRC)
    r = subprocess.run([build.HIPCC, "--cuda-host-only", "-O1", "-std=c++17", "-Wno-unused-function", "-I", build.CSRC,
                        str(tmp_path / "cols.hip"), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    spots = [(x, y) for x in (0, nx // 2, nx - 1, nx + 1, -2) for y in (0, ny // 2, ny - 1, ny + 1, -1)]

    def cell(g, n):  # the ghost rules of bound: periodic, or mirrored at the wall
        if bound == 2:
            return g % n
        return -1 - g if g < 0 else 2 * n - 1 - g if g >= n else g

    got = subprocess.run([str(exe), str(bound), str(nx), str(ny)] + [str(v) for s in spots for v in s],
                         capture_output=True, text=True, check=True).stdout.split()
    assert [int(v) for v in got] == [cell(x, nx) + nx * cell(y, ny) for x, y in spots]
