"""Launch grid of the z-marching columns (column.h): the planes per workgroup
are the cheapest of all, and finding them costs the host little.  Host code
only, no GPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <chrono>
#include <cstdio>
#include "column.h"
using namespace opsmi;

// the cost as column_grid's comment states it, over every chunk count
static int cheapest(const Range3 &r, int tile_x, int rows) {
  const ColGrid g = heat_column_grid(r, tile_x, rows);
  const long nz = r.z1 - r.z0, cus = inst().num_cus;
  long best = -1, chunk = 0;
  for (long k = (nz + 63) / 64; k <= nz; k++) {
    const long c = (nz + k - 1) / k, rounds = ((long)g.gx * g.gy * ((nz + c - 1) / c) + cus - 1) / cus;
    if (best < 0 || rounds * (c + 3) < best) best = rounds * (c + 3), chunk = c;
    if (c <= 2) break;
  }
  return (int)chunk;
}

template <class F>
static double nanoseconds(F f) {
  double best = 1e30;
  for (int rep = 0; rep < 7; rep++) {
    volatile int sink = 0;
    const auto t0 = std::chrono::steady_clock::now();
    for (int i = 0; i < 2000; i++) sink = sink + f().chunk;
    const double t = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count() / 2000 * 1e9;
    if (t < best) best = t;
  }
  return best;
}

int main() {
  inst().num_cus = 256;
  long bad = 0, seen = 0;
  for (int tile_x : {128, 256})
    for (int nx = 1; nx < 700; nx += 41)
      for (int ny = 1; ny < 700; ny += 37)
        for (int nz = 1; nz < 800; nz += 3, seen++) {
          const Range3 r{0, nx, 0, ny, 0, nz};
          const ColGrid g = column_grid(r, tile_x, 8);
          if (g.chunk != cheapest(r, tile_x, 8) || (long)g.gz != (nz + g.chunk - 1) / g.chunk) bad++;
        }
  printf("bad %ld of %ld\n", bad, seen);
  for (int n : {128, 256, 512}) {
    const Range3 r{0, n, 0, n, 0, n};
    printf("time %d %.1f %.1f\n", n, nanoseconds([&] { return heat_column_grid(r, 128, 8); }),
           nanoseconds([&] { return column_grid(r, 128, 8); }));
  }
}
"""


def test_cheapest_chunk_found_quickly(tmp_path):
    csrc = os.path.join(ROOT, "ops_amd", "csrc")
    src, exe, lib = tmp_path / "grid.hip", tmp_path / "grid", os.path.join(ROOT, "ops_amd")
    src.write_text(PROGRAM)
    subprocess.run(["hipcc", "-O2", "-std=c++17", "-x", "hip", "--offload-host-only", "-c", str(src), "-I", csrc,
                    "-o", str(tmp_path / "grid.o")], check=True)
    subprocess.run(["hipcc", str(tmp_path / "grid.o"), "-L", lib, "-lopsmi", "-Wl,-rpath," + lib, "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=120).stdout.splitlines()
    assert out[0].startswith("bad 0 of"), out[0]
    # 2 to 5 times the plain grid's few divisions (10 to 40 times when every
    # chunk count was tried)
    for line in out[1:]:
        _, n, plain, grid = line.split()
        assert float(grid) <= 8 * float(plain), line
