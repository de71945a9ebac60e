"""The step's field launches on the largest grids that a context accepts: no
dimension of 2^32 threads, every cell in one block, blocks past the last one
without a cell.  The launch shape is host arithmetic of a kernel header, here
compiled for the host alone."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCE = r"""
#include <stdio.h>
#include <stdlib.h>
#include "pic_fused.h"
int main(int argc, char **argv) {
  pic::Geom g = {};
  g.NX = atoi(argv[1]), g.NY = atoi(argv[2]), g.NZ = atoi(argv[3]);
  g.SX = g.NX + 4, g.SY = g.NY + 4, g.SZ = g.NZ + 4;
  const pic::CellBlocks cb(g);
  const int64_t n = cb.count(g);
  const dim3 d = pic::block_grid(n);
  printf("%lld %u %u %u\n", (long long)n, d.x, d.y, d.z);
  // the blocks around both ends and the middle, and those past the last one
  int64_t found = 0, past = 0;
  for (int64_t b = 0; b < (int64_t)d.x * d.y; ++b) {
    if (n > 4096 && b > 64 && (b < n / 2 || b > n / 2 + 64) && b < n - 64) continue;
    for (int t = 0; t < 256; ++t) {
      int k, l, m;
      if (!cb.cell(g, (int)b, t, k, l, m)) continue;
      if (k < 0 || l < 0 || m < 0 || k >= g.SX || l >= g.SY || m >= g.SZ) return 1;
      if (b >= n) ++past;
      ++found;
    }
  }
  const bool last = [&] {
    int k, l, m;
    return cb.cell(g, (int)(n - 1), ((g.SY - 1) % 4) * 64 + (g.SZ - 1) % 64, k, l, m) &&
           k == g.SX - 1 && l == g.SY - 1 && m == g.SZ - 1;
  }();
  printf("%lld %lld %d\n", (long long)found, (long long)past, (int)last);
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("grid")
    src, exe = d / "grid.hip", d / "grid"
    src.write_text(SOURCE)
    assert shutil.which(HIPCC)
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17",
                    "-I", os.path.join(ROOT, "plasmasim_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True)
    return str(exe)


# (8 x 8 x 16: every block; the others have up to 2^31 cells with the guards)
@pytest.mark.parametrize("n", [(8, 8, 16), (5, 7, 61), (8190, 8190, 8), (13370, 13370, 8),
                               (4, 22369000, 8), (1019, 1019, 1019)])
def test_field_launch_fits(program, n):
    out = subprocess.run([program, *map(str, n)], check=True, capture_output=True, text=True)
    blocks, x, y, z, found, past, last = map(int, out.stdout.split())
    cells = (n[0] + 4) * (n[1] + 4) * (n[2] + 4)
    assert cells <= 1 << 31
    assert x * y * z >= blocks and x * 256 < 1 << 32 and y <= 65535 and z == 1
    assert past == 0 and last == 1
    if blocks <= 4096:
        assert found == cells
