// Tile and offset arithmetic of the packed-row rel-pos kernel (attn_relpos_rows.hip): plain constexpr functions,
// so that a CPU program can walk every offset of every grid (tests/test_rows_offsets.py).
//
// A grid row is CPR chunks of 8 columns; tile t holds the chunks 8 t .. 8 t + 7 of a wave group's rows, which
// start at grid row r0. Offsets are in elements of the head.
#pragma once

namespace samhip {
namespace rows {

constexpr int gcd8(int c) { return c % 8 == 0 ? 8 : (c % 4 == 0 ? 4 : (c % 2 == 0 ? 2 : 1)); }
constexpr int period(int cpr) { return cpr / gcd8(cpr); }  // tiles after which the chunk pattern repeats

// The last chunk of a row from this one on reaches past the head's end in the last hd row: row W + 8 CPR > H W.
// It is the last row but for widths below 4, where the 8 columns of a chunk span several rows: H + 1 - ceil(8 / W)
// there (no division: its result would sit in a vector register).
constexpr int first_end_row(int H, int W, int cpr) {
  return H - (cpr > 1 || W > 3 ? 1 : W == 3 ? 2 : W == 2 ? 3 : 7);
}
// whether tile t holds a chunk of a row from `first` on
constexpr bool reaches_row(int t, int r0, int first, int cpr) { return 8 * t + 8 > (first - r0) * cpr; }

// first column of chunk j of the tile whose phase starts at chunk j0 of a row, in a row of hd (rows past the
// grid read the last one)
constexpr int k_column(int t, int j0, int kj, int r0, int H, int W, int cpr) {
  const int j = j0 + kj, add = j / cpr, cc = j - add * cpr;
  const int row = r0 + (8 * t) / cpr + add;
  return (row < H ? row : H - 1) * W + 8 * cc;
}
// elements by which the 8-element load of hd row d at column x starts early, to end with the head
constexpr int k_early(int d, int x, int N, int hd) {
  const int over = d * N + x + 8 - hd * N;
  return over > 0 ? over : 0;
}
// first V row of tile t in a group of `rows` grid rows: the range check of a buffer load subtracts the uniform
// offset from the buffer's size, so the tile past the last one (a prefetch) starts at the group's end, no later
constexpr int v_row(int t, int rows, int cpr) {
  const int r = 8 * t / cpr;
  return r < rows ? r : rows;
}

}  // namespace rows
}  // namespace samhip
