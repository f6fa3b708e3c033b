"""The walk over a result's tiles (csrc/walk.h): every launch it describes is one the device takes, and every tile is run once."""
import ctypes
import os
import subprocess

from swiftrt_amd import native

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include <vector>
#include "walk.h"
using namespace srt::waves;

// as the kernels divide
static uint32_t quotient(uint32_t n, uint32_t d, uint32_t rcp) { return rcp ? (uint32_t)(((uint64_t)n * rcp) >> 32) : n / d; }

static int launch_fits(int M, int N, int batch, int edge) {
  const uint64_t tiles = (uint64_t)((M + (int64_t)edge - 1) / edge) * ((N + (int64_t)edge - 1) / edge) * batch;
  const bool fits = (tiles + 7) / 8 * 8 * 256 < (1ull << 32);
  const Walk w = make_walk(M, N, batch, edge);
  if (w.tiles == (fits ? tiles : 0)) return 0;
  std::printf("%d %d %d %d: %u of %llu tiles\n", M, N, batch, edge, w.tiles, (unsigned long long)tiles);
  return 1;
}

static int covers(int M, int N, int batch, int edge, bool along_rows) {
  const Walk w = make_walk(M, N, batch, edge, along_rows);
  std::vector<char> seen(w.tiles, 0);
  for (uint32_t block = 0; block < 8 * w.chunk; ++block) {
    const uint32_t id = (block & 7) * w.chunk + (block >> 3);
    if (id >= w.tiles) continue;
    const uint32_t line = quotient(id, w.fast, w.fast_rcp), fast = id - line * w.fast;
    const uint32_t bz = quotient(line, w.slow, w.slow_rcp), slow = line - bz * w.slow;
    const uint32_t m = w.fast_is_m ? fast : slow, n = w.fast_is_m ? slow : fast, tm = (M + edge - 1) / edge, tn = (N + edge - 1) / edge;
    if (m >= tm || n >= tn || bz >= (uint32_t)batch || seen[(bz * tm + m) * tn + n]++) return 1;
  }
  for (char s : seen)
    if (!s) return 1;
  return 0;
}

int main() {
  int bad = 0;
  // the last count of tiles that one dimension of a grid holds, and the first that it does not, by rows, columns and matrices
  for (int edge : {32, 64, 128})
    for (long long t : {(1 << 24) - 9, (1 << 24) - 8, (1 << 24) - 7, 1 << 24, (1 << 24) + 1}) {
      if (t * edge <= 0x7fffffffLL) bad += launch_fits((int)(t * edge), 1, 1, edge) + launch_fits(1, (int)(t * edge), 1, edge);
      bad += launch_fits(1, (int)((t + 255) / 256 * edge), 256, edge) + launch_fits(3 * edge, (int)((t + 2) / 3 * edge), 1, edge);
    }
  bad += launch_fits(1, 8193, 65535, 32) + launch_fits(0x7fffffff, 0x7fffffff, 65535, 32) + launch_fits(0x7fffffff, 1, 1, 128);
  // quotients by multiplication up to 65535 tiles, by division past them; one row, one column
  const int shapes[][3] = {{1, 1, 1}, {33, 1, 5}, {1, 33, 5}, {1, 32 * 65535, 1}, {1, 32 * 65536, 1}, {32 * 255, 32 * 257, 1}, {97, 65, 5461},
                           {97, 65, 10923}, {33, 33, 16500}, {32 * 7, 32 * 13, 721}};
  for (const auto& s : shapes)
    for (bool along : {false, true})
      if (covers(s[0], s[1], s[2], 32, along)) {
        std::printf("%d x %d x %d: not every tile once\n", s[0], s[1], s[2]);
        ++bad;
      }
  return bad != 0;
}
"""


def test_walks_are_launches_and_cover_the_result(tmp_path):
    (tmp_path / "walk.cpp").write_text(DRIVER)
    exe = tmp_path / "walk"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "swiftrt_amd", "csrc"), "-o", str(exe),
                    str(tmp_path / "walk.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout


def test_rows_too_long_for_small_tiles_run_on_larger_ones():
    """2^24 tiles in one dimension of the grid are a launch the device refuses, by walk or by row."""
    buf, p = ctypes.create_string_buffer(64), ctypes.c_void_p(256)
    for M, tb in ((1, True), (8, False)):
        N, K = 1 << 29, 8
        bshape = (N, K) if tb else (K, N)
        ad, k1 = native.make_descriptor(native.REAL16BF, (M, K), (K, 1), native.ORDER_ROW)
        bd, k2 = native.make_descriptor(native.REAL16BF, bshape, (bshape[1], 1), native.ORDER_ROW)
        od, k3 = native.make_descriptor(native.REAL16BF, (M, N), (N, 1), native.ORDER_ROW)
        assert native.lib().srtMatmulQueryKernel(ctypes.byref(ad), 0, ctypes.byref(bd), int(tb), ctypes.byref(od), p, p, p, buf, 64) == 0
        assert buf.value.decode() == "mfma_128x128"
