"""Every offset that the packed-row rel-pos kernel (attn_relpos_rows.hip) loads from, walked on the CPU: a C++
program over its own tile arithmetic (rows_tiles.hpp) and every grid up to 64 x 64."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

K_LOADS = r"""
#include <cstdio>
#include "rows_tiles.hpp"
using namespace samhip::rows;

// The K loads of one wave group of gt threads: rows [r0, ..) of the grid, tiles 0 .. ntiles (the last is the
// prefetch of the loop's last step).
static int check(int H, int W, int hd, int gt, int r0, int ntiles) {
  const int cpr = (W + 7) / 8, N = H * W, first = first_end_row(H, W, cpr), rows = gt / 8;
  for (int t = 0; t <= ntiles; ++t) {
    const bool end = reaches_row(t, r0, first, cpr);
    for (int kj = 0; kj < 8; ++kj) {
      const int x = k_column(t, 8 * (t % period(cpr)) % cpr, kj, r0, H, W, cpr);
      for (int d = 0; d < hd; ++d) {
        if (d > 1 && d < hd - 8) continue;
        const int kd = d % rows, early = end ? k_early(d, x, N, hd) : 0, off = d * N + x - early;
        const bool whole = end || x + 8 <= N;  // else the 8 columns run into the next hd row uncleared
        if (off < 0 || off + 8 > hd * N || early > 7 || kd * N + x < early || !whole) {
          printf("H=%d W=%d hd=%d threads=%d r0=%d tile %d chunk %d d=%d: elements %d..%d of %d\n", H, W, hd, gt, r0,
                 t, kj, d, off, off + 7, hd * N);
          return 1;
        }
      }
    }
  }
  return 0;
}

int main() {
  int bad = 0;
  for (int hd = 64; hd <= 80; hd += 16)
    for (int H = 1; H <= 64; ++H)
      for (int W = 1; W <= 64; ++W) {
        const int cpr = (W + 7) / 8, half = (H + 1) / 2;
        bad += check(H, W, hd, 256, 0, (H * cpr + 7) / 8);  // one group of 4 waves
        bad += check(H, W, hd, 512, 0, (H * cpr + 7) / 8);  // one group of 8
        bad += check(H, W, hd, 256, 0, (half * cpr + 7) / 8);  // two groups of 4, the first and the second
        if (H > 1) bad += check(H, W, hd, 256, half, (half * cpr + 7) / 8);
      }
  printf("%d\n", bad);
  return bad != 0;
}
"""


V_LOADS = r"""
#include <cstdio>
#include "rows_tiles.hpp"
using namespace samhip::rows;

// The V loads of one wave group of `rows` grid rows, through a descriptor of rows * W * hd elements: the uniform
// offset must not pass its size (the check is offset >= size - uniform offset, and says nothing of a negative
// difference); slots past the row's W columns are sent out of range by the caller.
static int check(int H, int W, int hd, int rows, int ntiles) {
  const int cpr = (W + 7) / 8, size = rows * W * hd;
  for (int t = 0; t <= ntiles; ++t) {
    const int base = v_row(t, rows, cpr) * W * hd;
    bool ok = base <= size;
    for (int j = 0; j < 8 && ok; ++j) {
      const int chunk = 8 * t % cpr + j, add = chunk / cpr, cc = chunk % cpr, row = 8 * t / cpr + add;
      for (int c = 0; c < 8 && 8 * cc + c < W; ++c) {
        const int off = (add * W + 8 * cc + c) * hd;
        // a row of the group is read at its place, any other is out of range
        ok = ok && (row < rows ? base + off == (row * W + 8 * cc + c) * hd && off < size - base : off >= size - base);
      }
    }
    if (!ok) {
      printf("H=%d W=%d hd=%d rows=%d tile %d of %d: base %d, size %d\n", H, W, hd, rows, t, ntiles, base, size);
      return 1;
    }
  }
  return 0;
}

int main() {
  int bad = 0;
  for (int hd = 64; hd <= 80; hd += 16)
    for (int H = 1; H <= 64; ++H)
      for (int W = 1; W <= 64; ++W) {
        const int cpr = (W + 7) / 8, half = (H + 1) / 2;
        bad += check(H, W, hd, H, (H * cpr + 7) / 8);
        bad += check(H, W, hd, half, (half * cpr + 7) / 8);
        if (H > 1) bad += check(H, W, hd, H - half, (half * cpr + 7) / 8);
      }
  printf("%d\n", bad);
  return bad != 0;
}
"""


def run(tmp_path, source):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(source)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "sam-rs_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[:2000]


def test_k_loads_stay_in_the_head(tmp_path):
    run(tmp_path, K_LOADS)


def test_v_loads_stay_in_the_descriptor(tmp_path):
    run(tmp_path, V_LOADS)
