"""Launch shapes that no test can run at full size: compiled, not run (CPU
only; hipcc checks the assertions without generating code)."""
import os
import shutil
import subprocess

import pytest

from malus_amd import build as B

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

# HIP refuses 2^32 threads or more along x; the row kernels that give a row a
# workgroup of W threads have to cover any number of rows that fits the card.
ROWS = """
#include "k_rows.hip"
namespace malus {
namespace k {
namespace {
template <int W>
constexpr bool covers(size_t rows) {
  const dim3 g = RowLaunch<W>::grid(rows);
  return (size_t)g.x * RowLaunch<W>::threads < (1ull << 32) && g.y <= 65535 && g.z == 1 && (size_t)g.x * g.y >= rows &&
         (size_t)g.x * (g.y - 1) < rows;
}
template <int W>
constexpr bool edges() {
  constexpr size_t lim = (1ull << 32) / W;  // the first number of rows that one dimension does not take
  return covers<W>(1) && covers<W>(lim - 1) && covers<W>(lim) && covers<W>(lim + 1) && covers<W>(3 * lim + 7) &&
         RowLaunch<W>::grid(lim - 1).y == 1;
}
static_assert(edges<256>() && edges<512>() && edges<1024>(), "a row per workgroup");
}  // namespace
}  // namespace k
}  // namespace malus
"""


# A split GEMM's workgroups, dealt to eight XCDs round robin, take each entry
# of the work list once, every XCD one contiguous range.
XCD = """
#include "k_gemm_dma.h"
namespace malus {
namespace k {
constexpr bool ranges(int total) {
  bool seen[800] = {};
  for (int lin = 0; lin < total; ++lin) {
    const int w = xcd_range(lin, total);
    if (w < 0 || w >= total || seen[w]) return false;
    seen[w] = true;
    if (lin >= 8 && w != xcd_range(lin - 8, total) + 1) return false;
  }
  return true;
}
static_assert(ranges(1) && ranges(7) && ranges(8) && ranges(9) && ranges(36) && ranges(252) && ranges(255) &&
              ranges(256) && ranges(756) && ranges(799), "a list in eight ranges");
}  // namespace k
}  // namespace malus
"""


def compiles(tmp_path, text):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    src = tmp_path / "shape.hip"
    src.write_text(text)
    cmd = [HIPCC, "-x", "hip", *B.COMMON, *B.DEVICE, "--cuda-host-only", "-fsyntax-only", "-I", str(B.CSRC), str(src)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]


def test_rows_past_the_x_limit_of_a_launch(tmp_path):
    compiles(tmp_path, ROWS)


def test_work_list_in_eight_ranges(tmp_path):
    compiles(tmp_path, XCD)
