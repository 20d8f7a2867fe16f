"""Every byte the fp32 GEMM's tile loads read (triton-metal_amd/csrc/kernels/x3_runs.h,
compiled for the host): inside the operand where its rows are whole 16-byte runs, and
at most 12 bytes behind it elsewhere, where the planner asks for room."""

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "triton-metal_amd" / "csrc"

HARNESS = r'''
#include <cstdio>
#include <cstdlib>
#include <algorithm>
#include "kernels/x3_runs.h"
/* furthest byte read behind the last element of an operand of `rows` (CONTIG) or
 * columns times k, and the lowest byte read */
template <bool CONTIG> void walk(int tile, int64_t ld, int rows, int k, long long &past, long long &low) {
  const long long end = 4 * (CONTIG ? (rows - 1) * ld + k : (k - 1) * ld + rows);
  for (int r0 = 0; r0 < rows; r0 += tile)
    for (int k0 = 0; k0 < k; k0 += 32) {
      const long long base = 4 * (CONTIG ? r0 * ld + k0 : k0 * ld + r0);
      const int left = std::min(rows - r0, tile), k_left = k - k0;
      for (int row = 0; row < (CONTIG ? tile : 32); ++row)
        for (int col = 0; col < (CONTIG ? 32 : tile); col += 4) {
          uint32_t run = x3_run<CONTIG>(ld, row, col, left);
          if (k_left < 32) run = x3_last_run<CONTIG>(run, ld, row, col, k_left);
          past = std::max(past, base + run + 16 - end);
          low = std::min(low, base + (long long)run);
        }
    }
}
int main(int, char **v) {
  long long past = -(1LL << 60), low = 1LL << 60;
  const int tile = atoi(v[2]), rows = atoi(v[4]), k = atoi(v[5]);
  const int64_t ld = atoll(v[3]);
  if (atoi(v[1])) walk<true>(tile, ld, rows, k, past, low);
  else walk<false>(tile, ld, rows, k, past, low);
  printf("%lld %lld\n", past, low);
}
'''

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@pytest.fixture(scope="module")
def reads(tmp_path_factory):
    d = tmp_path_factory.mktemp("x3_runs")
    (d / "h.cpp").write_text(HARNESS)
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{CSRC}", str(d / "h.cpp"), "-o", str(d / "h")], check=True)

    def run(contig, tile, ld, rows, k):
        out = subprocess.run([str(d / "h"), *map(str, (int(contig), tile, ld, rows, k))],
                             check=True, capture_output=True, text=True).stdout
        return tuple(map(int, out.split()))
    return run


@pytest.mark.parametrize("contig", [True, False])
@pytest.mark.parametrize("tile", [64, 128])
@pytest.mark.parametrize("rows,k", [(64, 64), (192, 96), (320, 512), (1088, 64), (68, 36), (4, 36), (132, 100)])
def test_whole_runs_stay_inside(reads, contig, tile, rows, k):
    """Sizes of whole 16-byte runs, tiles part empty among them: nothing behind the
    operand is read, with rows as long as the matrix or longer."""
    for ld in ((k, k + 8) if contig else (rows, rows + 8)):
        past, low = reads(contig, tile, ld, rows, k)
        assert past <= 0 and low == 0, (ld, past, low)


@pytest.mark.parametrize("contig", [True, False])
@pytest.mark.parametrize("tile", [64, 128])
@pytest.mark.parametrize("rows,k", [(1, 33), (65, 63), (129, 97), (255, 130), (3, 65), (66, 34)])
def test_other_sizes_read_at_most_12_bytes_behind(reads, contig, tile, rows, k):
    for pad in (0, 1):
        past, low = reads(contig, tile, (k if contig else rows) + pad, rows, k)
        assert past <= 12 and low == 0, (pad, past, low)


@pytest.mark.parametrize("m,n,k,layout,clipped", [
    (2048, 1088, 8192, "nn", 1088), (1088, 2048, 8192, "tn", 1088)
])
def test_whole_tiles_of_64_on_the_128_kernel(reads, m, n, k, layout, clipped):
    """fp32 products of whole 64 x 64 tiles, an operand exactly filling buffers of
    whole 2 MiB (nothing behind them), which run 128 x 128 tiles."""
    import planner
    from test_planner import _matmul
    if not planner.buildable():
        pytest.skip("built code objects absent")
    assert clipped * k * 4 % (2 << 20) == 0
    planner.launched()
    _matmul("f32", layout, m, n, k)
    assert planner.launched()[0][0] == f"tm_gemm_x3{'_tn' if layout == 'tn' else ''}_f32"
    past, _ = reads(False, 128, clipped, clipped, k)
    assert past <= 0
