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


def test_rows_past_the_x_limit_of_a_launch(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    src = tmp_path / "rows.hip"
    src.write_text(ROWS)
    cmd = [HIPCC, "-x", "hip", *B.COMMON, *B.DEVICE, "--cuda-host-only", "-fsyntax-only", "-I", str(B.CSRC), str(src)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]
