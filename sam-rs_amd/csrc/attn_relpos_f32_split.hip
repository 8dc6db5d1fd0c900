// Fused rel-pos attention in f32 at hd 64 and 80 for grids up to 64 x 64, on the bf16 matrix units, for gfx950.
//
//   out[bh, r, :] = softmax_k( scale * q[r] . k[k] + q[r] . Th[i - kh + H-1] + q[r] . Tw[j - kw + W-1] ) . v
//
// An f32 is the sum of three bf16 terms (8 + 8 + 8 bits of mantissa), so an f32 product is six bf16 products,
// hi.hi, hi.mid, mid.hi, mid.mid, hi.lo and lo.hi, summed in f32; the three that are left out are below 2^-24
// of it. q, k, v, the table and the softmax weights are all taken so: nothing is held in fewer bits than f32.
// The f32 MFMA runs at 1/16 of the bf16 rate, so six of these take 3/8 of its time.
//
// Layouts are those of attn_relpos_rows.hip: S^T = K . Q^T on 32 x 32 x 16 tiles with one query per lane,
// O^T = V^T . P^T straight from the S^T accumulators, grid rows padded to a multiple of 8 columns (CPR chunks
// of 8) that are packed into tiles of 32 slots, Rw in 4 CPR registers, Rh from LDS. K and V are read as f32,
// split once per workgroup while they are stored to LDS (three planes each) and read with transpose reads.
//   * K planes [hd][32 slots], 64-byte rows, and V planes [32 slots][hd]: four consecutive rows of 32 elements
//     fall on all 64 banks (hd 64: the 32-column halves of rows 2, 3 mod 4 are swapped for that).
//   * the softmax runs in the exp2 domain: u = s * (scale log2e) + (rh - m) + rw, one fma and one add a score.
//   * a tile's weights are summed by themselves and then added to the running sum, so the rounding of a long
//     row's denominator grows with its tiles; the products go straight into the running O.
//   * G = 2: two groups of waves take half of the grid rows each for the same queries and merge at the end.
// An infinity splits into inf - inf, and what a low term has below 2^-133 is lost (of values below 2^-110 some of
// the 24 bits: v of about 2^-120 gave 9e-5 of relative error). So a row with a result that is not finite, or not 0
// and below 2^-104, is computed again on the f32 matrix units (relpos_f32_rows): infinities, NaN and small values
// come out as f32 arithmetic has them. In a score the loss is 2^-133 of the other factor.
#include <type_traits>

#include "common.hpp"
#include "relpos_geom.hpp"

namespace samhip {

namespace f32s {

constexpr float kSlack = 8.0f;  // log2 units by which a weight may exceed 1 before the maximum moves
// least result that the three terms hold in full: what they lose is below 2^-133, the last bit of a small bf16
constexpr unsigned kLeastHeld = (127 - 104) << 23;  // 2^-104

template <int HD> struct Shape {
  static constexpr int kKS = HD / 16;
  static constexpr int kMBO = (HD + 31) / 32;
  static constexpr int kVS = HD;                      // elements of a V plane's row
  static constexpr int kKPlane = HD * 32, kVPlane = 32 * kVS;
  static constexpr int kBuf = 3 * (kKPlane + kVPlane);  // elements of one tile
};

// 4-wave workgroups at hd 64 hold up to 5 chunks a row in 168 registers, so that three share a CU
constexpr int waves_per_simd(int hd, int cpr, int qw, int g) { return hd == 64 && cpr <= 5 && qw * g == 4 ? 3 : 2; }

constexpr int gcd4(int c) { return c % 4 == 0 ? 4 : (c % 2 == 0 ? 2 : 1); }
constexpr int period(int cpr) { return cpr / gcd4(cpr); }  // tiles after which the chunk pattern repeats

__device__ __forceinline__ int xcd_block(int i, int total) {
  const int per = total >> 3, rem = total & 7, x = i & 7, j = i >> 3;
  return x * per + (x < rem ? x : rem) + j;
}

// x = hi + mid + lo, exact for every finite x whose low term keeps its bits (|x| from 2^-110 on). Two at a time on
// the packed conversion; the terms go back to f32 by a shift and a mask.
struct Split {
  bf16x8 t[3];
};
__device__ __forceinline__ Split split3(const float* x) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef bf16 bf16x2 __attribute__((ext_vector_type(2)));
  u32x4 r[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float y0 = x[2 * i], y1 = x[2 * i + 1];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const unsigned u = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{y0, y1}, bf16x2));
      r[p][i] = u;
      y0 -= __uint_as_float(u << 16);
      y1 -= __uint_as_float(u & 0xffff0000u);
    }
  }
  Split s;
#pragma unroll
  for (int p = 0; p < 3; ++p) s.t[p] = __builtin_bit_cast(bf16x8, r[p]);
  return s;
}

// acc += a . b over the six products that f32 holds; the small ones first, which helps where acc starts small (S^T)
__device__ __forceinline__ f32x16 mma6(const bf16x8* a, const bf16x8* b, f32x16 acc) {
  acc = mma32(a[2], b[0], acc);
  acc = mma32(a[0], b[2], acc);
  acc = mma32(a[1], b[1], acc);
  acc = mma32(a[1], b[0], acc);
  acc = mma32(a[0], b[1], acc);
  return mma32(a[0], b[0], acc);
}

}  // namespace f32s

// The 32 queries of a wave (from q0, one a lane of either half) on the f32 matrix units, straight from memory:
// 32 keys of one grid row a tile, logits (q . k) * scale + rh + rw, accurate expf. rhs is the wave's own bias
// scratch, rows of 32. Only the rows in `bad` are stored. Nothing is staged: bound by the latency of its loads. With a
// NaN in every head, 12 heads of 64 x 64 at hd 64 take 1.24 ms (0.33 clean; the f32 MFMA kernel before 0.6; one wave
// a row in plain f32, as this was first done, 42), 300 windows of 14 x 14 0.19 (2.3).
template <int HD>
__device__ __forceinline__ void relpos_f32_rows(const float* __restrict__ q, const float* __restrict__ kt,
                                                const float* __restrict__ v, const float* __restrict__ table,
                                                float* __restrict__ out, float* rhs, int q0, unsigned bad, int H, int W,
                                                float scale) {
  constexpr int kHalf = HD / 2, kMBO = (HD + 31) / 32;  // k-step s takes dims s (lower lanes) and kHalf + s (upper)
  constexpr float kSlackNat = 5.5451774f;               // 8 ln 2
  const int lane = threadIdx.x & 63, n = lane & 31, hh = lane >> 5, N = H * W;
  const int qidx = min(q0 + n, N - 1), qi = qidx / W, qj = qidx % W;
  auto wsync = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  float qf[kHalf];
#pragma unroll
  for (int s = 0; s < kHalf; s += 4) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(q + (long)qidx * HD + kHalf * hh + s);
#pragma unroll
    for (int e = 0; e < 4; ++e) qf[s + e] = x[e];
  }
  // rhs[k] = q . tab[base - k + len - 1]
  auto band = [&](const float* tab, int base, int len) {
    wsync();
    for (int b = 0; b < 2 * len - 1; b += 32) {
      const float* trow = tab + (long)min(b + n, 2 * len - 2) * HD + kHalf * hh;
      f32x16 acc = {};
#pragma unroll
      for (int s = 0; s < kHalf; s += 4) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(trow + s);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], qf[s + e], acc, 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int k = base + len - 1 - b - (8 * (e >> 2) + 4 * hh + (e & 3));
        if (k >= 0 && k < len) rhs[k * 32 + n] = acc[e];
      }
    }
    wsync();
  };
  float m = -INFINITY, l = 0.f;
  f32x16 o[kMBO];
#pragma unroll
  for (int ob = 0; ob < kMBO; ++ob) o[ob] = f32x16{};
  for (int c0 = 0; c0 < W; c0 += 32) {
    band(table + (long)(2 * H - 1) * HD, qj, W);
    float rw[16];  // columns c0 + 8 (e / 4) + 4 hh + e % 4
#pragma unroll
    for (int e = 0; e < 16; ++e) rw[e] = rhs[min(c0 + 8 * (e >> 2) + 4 * hh + (e & 3), W - 1) * 32 + n];
    band(table, qi, H);
    for (int row = 0; row < H; ++row) {
      unsigned col0 = c0 + 4 * hh;  // as the asm leaves it: what follows is computed here, not held for every row
      asm volatile("" : "+v"(col0));
      const float* kcol = kt + (long)kHalf * hh * N + row * W + min(c0 + n, W - 1);
      f32x16 s = {};
#pragma unroll
      for (int d = 0; d < kHalf; ++d) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kcol[(long)d * N], qf[d], s, 0, 0, 0);
      const float rh = rhs[row * 32 + n];
      float mm = -INFINITY;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float x = s[e] * scale + rh + rw[e];
        s[e] = (int)col0 + 8 * (e >> 2) + (e & 3) < W ? x : -INFINITY;
        mm = fmaxf(mm, s[e]);
      }
      const float mt = max_with_partner32(mm);
      if (wave_any(mt > m + kSlackNat)) {
        const float m_new = fmaxf(m, mt);
        const float alpha = m == -INFINITY ? 0.f : expf(m - m_new);
        l *= alpha;
#pragma unroll
        for (int ob = 0; ob < kMBO; ++ob) o[ob] *= alpha;
        m = m_new;
      }
      const float c = m == -INFINITY ? 0.f : m;  // all scores so far -inf: weight 0
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        s[e] = expf(s[e] - c);
        l += s[e];
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int col = (int)col0 + 8 * (e >> 2) + (e & 3);
        const unsigned voff = (unsigned)((row * W + min(col, W - 1)) * HD);
#pragma unroll
        for (int ob = 0; ob < kMBO; ++ob) {
          const float a = v[voff + (unsigned)min(32 * ob + n, HD - 1)];
          o[ob] = __builtin_amdgcn_mfma_f32_32x32x2f32(col < W ? a : 0.f, s[e], o[ob], 0, 0, 0);
        }
      }
    }
  }
  const float inv = 1.f / sum_with_partner32(l);
  if ((bad >> n) & 1) {
    float* orow = out + (long)(q0 + n) * HD;
#pragma unroll
    for (int ob = 0; ob < kMBO; ++ob)
#pragma unroll
      for (int a = 0; a < 4; ++a)
        if (32 * ob + 8 * a < HD)
          *reinterpret_cast<f32x4*>(orow + 32 * ob + 8 * a + 4 * hh) =
              f32x4{o[ob][4 * a] * inv, o[ob][4 * a + 1] * inv, o[ob][4 * a + 2] * inv, o[ob][4 * a + 3] * inv};
  }
}

// QW waves of 32 queries in each of G groups; NB tile buffers a group (2: one barrier a tile; 1: two, for
// workgroups that share a CU). Bound by the matrix units: 16 heads of 64 x 64 at hd 64 are 412 GFLOP of bf16
// products in 334 us, 1.23 PFLOP/s, what a large bf16 GEMM reaches on the card (1.19). The f32 MFMA kernel
// before it took 695 us (16 heads), 530 (12 heads, now 281), and 67 for 300 windows of 14 x 14 (now 37).
template <int HD, int CPR, int QW, int G, int NB>
__global__ __launch_bounds__(QW* G * 64, f32s::waves_per_simd(HD, CPR, QW, G)) void attn_relpos_f32_split_kernel(
    const float* __restrict__ q, const float* __restrict__ kt, const float* __restrict__ v,
    const float* __restrict__ table, float* __restrict__ out, int H, int W, float scale, float sc, int qblocks) {
  using namespace f32s;
  typedef Shape<HD> S;
  constexpr int kKS = S::kKS, kMBO = S::kMBO, kVS = S::kVS;
  constexpr int kGT = QW * 64;  // threads of a group
  constexpr int U = period(CPR);

  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qw = wave % QW, grp = wave / QW;
  const int gt = tid % kGT;
  bf16* gbase = reinterpret_cast<bf16*>(smem) + grp * NB * S::kBuf;
  const int R = H > W ? H : W;
  // per query wave: [row or column][query lane]; row R takes discarded scatters
  float* rhs = reinterpret_cast<float*>(reinterpret_cast<bf16*>(smem) + G * NB * S::kBuf) + qw * (R + 1) * 32;

  const int N = H * W;
  const int n = lane & 31, hh = lane >> 5, g4 = lane >> 4, gi = lane & 15;
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  const long bh = blk / qblocks;
  const int q0 = (blk % qblocks) * (QW * 32) + qw * 32;
  const bool active = q0 < N;  // whole wave
  const int qidx = q0 + n;
  const bool qvalid = qidx < N;
  const int qi = qvalid ? qidx / W : 0, qj = qvalid ? qidx % W : 0;

  // grid rows [r0, r1) of this group, and the tiles of the larger group (the first)
  const int hsplit = G == 1 ? H : (H + 1) / 2;
  const int r0 = grp == 0 ? 0 : hsplit, r1 = grp == 0 ? hsplit : H;
  const int ntiles = (hsplit * CPR + 3) / 4;

  // ---- staging. Tile t holds the chunks 4 t .. 4 t + 3. K: 8 columns of hd row d; columns past W are the
  // next grid row's keys, masked by the bias. V: 8 dims of a slot; slots past W or r1 are zero. Buffer loads
  // give zeros past the head's end, and for the offset that stands for a row past the grid.
  constexpr int kKItems = HD * 4, kVItems = 32 * (HD / 8);
  constexpr int KPT = (kKItems + kGT - 1) / kGT, VPT = (kVItems + kGT - 1) / kGT;
  constexpr int kOut = 0x40000000;
  float kreg[KPT][8], vreg[VPT][8];
  const auto krsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(kt + bh * HD * (long)N), 0,
                                                       (int)(HD * N * sizeof(float)), 0x00020000);
  const auto vrsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(v + bh * HD * (long)N), 0,
                                                       (int)(HD * N * sizeof(float)), 0x00020000);
  // At hd 80 the remainder of items goes to the first waves for K and to the last ones for V (16 heads of 37 x 50 132 us,
  // 135 with both to the first). At hd 64, where 8 waves have half a round of each, the first four take both (12 heads
  // of 64 x 64 282 us; 291 with V to the last four).
  constexpr bool kFar = HD == 80 && kVItems % kGT != 0;
  auto kitem = [&](int u) { return gt + u * kGT; };
  auto vitem = [&](int u) { return (kFar ? kGT - 1 - gt : gt) + u * kGT; };
  auto kin = [&](int u) { return kKItems % kGT == 0 || u + 1 < KPT || kitem(u) < kKItems; };
  auto vin = [&](int u) { return kVItems % kGT == 0 || u + 1 < VPT || vitem(u) < kVItems; };
  auto load8 = [&](auto rsrc, int off, float* x) {
    const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0);
    const u32x4 b = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off + 16, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[i] = __uint_as_float(a[i]);
      x[4 + i] = __uint_as_float(b[i]);
    }
  };
  auto load = [&](int t) {
#pragma unroll
    for (int u = 0; u < KPT; ++u) {
      const int c = 4 * t + (kitem(u) & 3), row = r0 + c / CPR, cc = c % CPR;
      const int off = row < H ? (int)(((kitem(u) >> 2) * N + row * W + 8 * cc) * sizeof(float)) : kOut;
      if (kin(u)) load8(krsrc, off, kreg[u]);
    }
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
      const int it = vitem(u), sl = it / (HD / 8);
      const int c = 4 * t + (sl >> 3), row = r0 + c / CPR, col = 8 * (c % CPR) + (sl & 7);
      const bool ok = row < r1 && col < W;
      const int off = ok ? (int)(((row * W + col) * HD + 8 * (it % (HD / 8))) * sizeof(float)) : kOut;
      if (vin(u)) load8(vrsrc, off, vreg[u]);
    }
  };
  // hd 64: the two 32-column halves of a V row change places in rows 2, 3 (mod 4)
  auto vcol = [&](int row, int col) { return HD == 64 ? col ^ (32 * ((row >> 1) & 1)) : col; };
  auto store = [&](int t) {
    bf16* kb = gbase + (NB == 2 ? t & 1 : 0) * S::kBuf;
    bf16* vb = kb + 3 * S::kKPlane;
#pragma unroll
    for (int u = 0; u < KPT; ++u) {
      if (kin(u)) {
        const Split s = split3(kreg[u]);
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8*>(kb + p * S::kKPlane + kitem(u) * 8) = s.t[p];
      }
    }
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
      if (vin(u)) {
        const Split s = split3(vreg[u]);
        const int sl = vitem(u) / (HD / 8), col = vcol(sl, 8 * (vitem(u) % (HD / 8)));
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8*>(vb + p * S::kVPlane + sl * kVS + col) = s.t[p];
      }
    }
  };

  // ---- prologue: the first tile in flight, q fragments, the bias bands
  load(0);
  bf16x8 qf[kKS][3];
  {
    const float* qrow = q + (bh * N + (qvalid ? qidx : 0)) * HD;
#pragma unroll
    for (int s = 0; s < kKS; ++s) {
      const Split x = split3(qrow + 16 * s + 8 * hh);
#pragma unroll
      for (int p = 0; p < 3; ++p) qf[s][p] = x.t[p];
    }
  }
  // The bias bands: G = T . Q^T in 32-row blocks, scattered along the diagonal in log2 units (entries outside
  // the band go to rows that are not read, or to the junk row). The table is split once for the workgroup,
  // into the tile buffers: whole if it fits, as a window's does, or kCap rows at a time.
  constexpr int kTS = HD == 64 ? 72 : HD;  // row stride: 8 rows' 16-byte reads fall on different banks
  constexpr int kCap = G * NB * S::kBuf / (3 * kTS), kCap32 = kCap / 32 * 32;
  bf16* tbl = reinterpret_cast<bf16*>(smem);
  const bool whole = 2 * (H + W) - 2 <= kCap;
  auto stage_table = [&](int row0, int rows) {
    for (int c = tid; c < rows * (HD / 8); c += QW * G * 64) {
      const int r = c / (HD / 8), d = 8 * (c % (HD / 8));
      const Split x = split3(table + (long)(row0 + r) * HD + d);
#pragma unroll
      for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8*>(tbl + (p * kCap + r) * kTS + d) = x.t[p];
    }
    __syncthreads();
  };
  auto band = [&](int row0, int nrows, int base, int len, bool mine) {
    const int top = base + len - 1 - 4 * hh;  // kh = i + H-1 - row, kw = j + W-1 - row
    for (int c0 = 0; c0 < nrows; c0 += kCap32) {
      if (!whole) stage_table(row0 + c0, min(kCap32, nrows - c0));
      if (mine) {
        const int end = min(nrows - c0, kCap32);
        for (int b = 0; b < end; b += 32) {
          f32x16 acc = {};
          const bf16* trow = tbl + ((whole ? row0 + c0 : 0) + min(b + n, end - 1)) * kTS + 8 * hh;
#pragma unroll
          for (int s = 0; s < kKS; ++s) {
            bf16x8 a[3];
#pragma unroll
            for (int p = 0; p < 3; ++p) a[p] = *reinterpret_cast<const bf16x8*>(trow + p * kCap * kTS + 16 * s);
            acc = mma6(a, qf[s], acc);
          }
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const unsigned k = (unsigned)(top - c0 - b - (8 * (e >> 2) + (e & 3)));
            rhs[min(k, (unsigned)R) * 32 + n] = acc[e] * kLog2e;
          }
        }
      }
      if (!whole) __syncthreads();
    }
  };
  if (whole) stage_table(0, 2 * (H + W) - 2);
  band(2 * H - 1, 2 * W - 1, qj, W, active && grp == 0);
  __syncthreads();
  float rw[4 * CPR];  // this lane's columns 8 cc + 4 hh + b
#pragma unroll
  for (int cc = 0; cc < CPR; ++cc)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int col = 8 * cc + 4 * hh + b;
      const float x = rhs[(col < W ? col : 0) * 32 + n];
      rw[4 * cc + b] = col < W ? x : -INFINITY;
    }
  __syncthreads();
  band(0, 2 * H - 1, qi, H, active && grp == G - 1);
  if (whole) __syncthreads();
  store(0);
  __syncthreads();

  // per-lane offsets of the transpose reads; planes, k-steps and blocks are constants added to them
  const int kl = (8 * (g4 >> 1) + (gi >> 2)) * 32 + 16 * (g4 & 1) + 4 * (gi & 3);
  const int vrow = 4 * (g4 >> 1) + (gi >> 2);
  int vl[kMBO];
#pragma unroll
  for (int ob = 0; ob < kMBO; ++ob) vl[ob] = vrow * kVS + vcol(vrow, 32 * ob) + 16 * (g4 & 1) + 4 * (gi & 3);

  float m_run = 0.f, l_run = 0.f;
  f32x16 o[kMBO];
#pragma unroll
  for (int ob = 0; ob < kMBO; ++ob) o[ob] = f32x16{};

  auto step = [&](int t, auto uc) {
    constexpr int j0 = (4 * decltype(uc)::value) % CPR;
    if (t + 1 < ntiles) load(t + 1);
    if (active) {
      const bf16* kb = gbase + (NB == 2 ? t & 1 : 0) * S::kBuf;
      const bf16* vb = kb + 3 * S::kKPlane;
      f32x16 s = {};
#pragma unroll
      for (int k = 0; k < kKS; ++k) {
        bf16x8 a[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          const bf16* x = kb + kl + p * S::kKPlane + 16 * k * 32;
          a[p] = join8<bf16>(lds_read_tr16(x), lds_read_tr16(x + 4 * 32));
        }
        s = mma6(a, qf[k], s);
      }
      float rh[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j == 0 || (j0 + j) % CPR == 0) {
          const int row = r0 + (4 * t) / CPR + (j0 + j) / CPR;
          const float x = rhs[(row < r1 ? row : r0) * 32 + n];
          rh[j] = row < r1 ? x - m_run : -INFINITY;
        } else {
          rh[j] = rh[j - 1];
        }
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = fmaf(s[e], sc, rh[e >> 2]) + rw[4 * ((j0 + (e >> 2)) % CPR) + (e & 3)];
      float mm = s[0];
#pragma unroll
      for (int e = 1; e < 16; ++e) mm = max_nc(mm, s[e]);
      const float mt = max_with_partner32(mm);
      if (t == 0 || wave_any(mt > kSlack)) {
        const float delta = t == 0 ? mt : max_nc(mt, 0.f);
        const float alpha = t == 0 ? 1.f : exp2_fast(-delta);
        m_run += delta;
        l_run *= alpha;
#pragma unroll
        for (int ob = 0; ob < kMBO; ++ob) o[ob] *= alpha;
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] -= delta;
      }
      float ls[4] = {0.f, 0.f, 0.f, 0.f};
      Split b[2];
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        float pv[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          pv[e] = exp2_fast(s[8 * w + e]);
          ls[e & 3] += pv[e];
        }
        b[w] = split3(pv);
      }
      l_run += (ls[0] + ls[1]) + (ls[2] + ls[3]);
#pragma unroll
      for (int ob = 0; ob < kMBO; ++ob) {
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          bf16x8 a[3];
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            const bf16* x = vb + vl[ob] + p * S::kVPlane + 16 * w * kVS;
            a[p] = join8<bf16>(lds_read_tr16(x), lds_read_tr16(x + 8 * kVS));
          }
          o[ob] = mma6(a, b[w].t, o[ob]);
        }
      }
    }
    if constexpr (NB == 1) __syncthreads();  // every wave is done with tile t
    if (t + 1 < ntiles) store(t + 1);
    __syncthreads();
  };

  for (int t = 0; t < ntiles; t += U) {
    step(t, std::integral_constant<int, 0>());
#define SAMHIP_STEP(i)   \
  if constexpr ((i) < U) \
    if (t + (i) < ntiles) step(t + (i), std::integral_constant<int, (i) % U>());
    SAMHIP_STEP(1)
    SAMHIP_STEP(2)
    SAMHIP_STEP(3)
    SAMHIP_STEP(4)
    SAMHIP_STEP(5)
    SAMHIP_STEP(6)
#undef SAMHIP_STEP
  }

  float l = sum_with_partner32(l_run);
  if constexpr (G == 2) {
    // the second group hands over O, max and sum; the last step's barrier freed the tile buffers
    float* xch = reinterpret_cast<float*>(smem) + qw * (16 * kMBO + 2) * 64;
    if (grp == 1) {
#pragma unroll
      for (int ob = 0; ob < kMBO; ++ob)
#pragma unroll
        for (int a = 0; a < 4; ++a)
          *reinterpret_cast<f32x4*>(xch + ((ob * 4 + a) * 64 + lane) * 4) =
              f32x4{o[ob][4 * a], o[ob][4 * a + 1], o[ob][4 * a + 2], o[ob][4 * a + 3]};
      xch[16 * kMBO * 64 + lane] = m_run;
      xch[(16 * kMBO + 1) * 64 + lane] = l;
    }
    __syncthreads();
    if (grp == 1) return;
    const float m1 = xch[16 * kMBO * 64 + lane], l1 = xch[(16 * kMBO + 1) * 64 + lane];
    const float M = max_nc(m_run, m1);
    const float w0 = exp2_fast(m_run - M), w1 = exp2_fast(m1 - M);
    l = l * w0 + l1 * w1;
#pragma unroll
    for (int ob = 0; ob < kMBO; ++ob)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(xch + ((ob * 4 + a) * 64 + lane) * 4);
#pragma unroll
        for (int b = 0; b < 4; ++b) o[ob][4 * a + b] = o[ob][4 * a + b] * w0 + x[b] * w1;
      }
  }

  // ---- normalise and store: lane holds O^T[32*ob + 8*a + 4*hh + b][query n]
  const float inv = 1.f / l;
  unsigned least = ~0u;  // of 2 |bits| - 1, which puts 0 last
  float most = 0.f;
  if (qvalid) {
    float* orow = out + (bh * N + qidx) * HD;
#pragma unroll
    for (int ob = 0; ob < kMBO; ++ob)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        if (32 * ob + 8 * a < HD) {
          f32x4 w4;
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            w4[b] = o[ob][4 * a + b] * inv;
            least = min(least, 2 * __float_as_uint(w4[b]) - 1);
            most = max_nc(most, __builtin_fabsf(w4[b]));
          }
          *reinterpret_cast<f32x4*>(orow + 32 * ob + 8 * a + 4 * hh) = w4;
        }
      }
  }
  unsigned long bad = __builtin_amdgcn_ballot_w64(least < 2 * kLeastHeld - 1 || !(most < INFINITY));
  bad = (bad | (bad >> 32)) & 0xffffffffu;
  // The same wave as the stores above, so later in order; rhs is this wave's alone by now. Never expected: otherwise
  // the compiler gives up registers of the key loop for it (109 heads of 29 x 16 at hd 80 58.7 us without these rows'
  // code, 64.8 with it, 59.6 so).
  if (__builtin_expect_with_probability(bad != 0, 0, 1.0))
    relpos_f32_rows<HD>(q + bh * HD * (long)N, kt + bh * HD * (long)N, v + bh * HD * (long)N, table,
                        out + bh * HD * (long)N, rhs, q0, (unsigned)bad, H, W, scale);
}

template <int HD, int CPR, int QW, int G, int NB>
static hipError_t launch_f32_split(const void* q, const void* kt, const void* v, const void* table, void* out, int bh,
                                   int h, int w, float scale, hipStream_t stream) {
  typedef f32s::Shape<HD> S;
  constexpr size_t tiles = (size_t)G * NB * S::kBuf * sizeof(bf16);
  constexpr size_t most = tiles + QW * 65 * 32 * sizeof(float);
  static_assert(most <= 160 * 1024, "LDS");
  static_assert(G == 1 || QW * (16 * S::kMBO + 2) * 64 * sizeof(float) <= tiles, "the exchange must fit");
  auto kern = attn_relpos_f32_split_kernel<HD, CPR, QW, G, NB>;
  static std::atomic<unsigned long long> lds_done{0};
  if (const hipError_t e = lds_opt_in(lds_done, (const void*)kern, (int)most); e != hipSuccess) return e;
  const int r = h > w ? h : w;
  const size_t lds = tiles + (size_t)QW * (r + 1) * 32 * sizeof(float);
  const int qblocks = (h * w + QW * 32 - 1) / (QW * 32);
  hipLaunchKernelGGL(kern, dim3((unsigned)(bh * qblocks)), dim3(QW * G * 64), lds, stream, (const float*)q,
                     (const float*)kt, (const float*)v, (const float*)table, (float*)out, h, w, scale,
                     (float)((double)scale * 1.4426950408889634), qblocks);
  return hipGetLastError();
}

// Which workgroup: 128 queries on 4 waves (two or three of them share a CU), 128 queries on two groups of 4
// waves that take half of the keys each, or 256 queries on 8 waves. The time is that of the fullest CU, in us
// at hd 64 as measured: a tile of 32 slots takes a SIMD's two waves 2.8 when every 4 waves stage their own
// keys, 2.6 when 8 share them, and a wave that has its SIMD to itself 2.0; a round costs about 5 beside its
// tiles. (The kernel has become 10-20% faster than these since they were fitted, in all three forms.) Measured
// (4 waves / two groups / 8 waves): 300 heads of 14 x 14 37 / 53 / 48, 12 of 64 x 64 328 / 333 / 281, 24 of 33 x 37
// 92 / 70 / 104, 96 of 12 x 12 18.2 / 16.5 / 20.2; at hd 80 16 of 37 x 50 186 / 141 / 207, 96 of 30 x 30
// 187 / 188 / 202, 16 of 48 x 56 302 / 315 / 262.
template <int HD, int CPR>
static hipError_t f32_split_waves(const void* q, const void* kt, const void* v, const void* table, void* out, int bh,
                                  int h, int w, float scale, hipStream_t stream) {
  const int cus = device_cu_count(), n = h * w;
  const long b4 = (long)bh * ((n + 127) / 128), b8 = (long)bh * ((n + 255) / 256);
  const long r4 = (b4 + cus - 1) / cus, r8 = (b8 + cus - 1) / cus;
  const float tile = HD / 64.f * ((h * CPR + 3) / 4), half = HD / 64.f * (((h + 1) / 2 * CPR + 3) / 4);
  const float four = (r4 / 2) * (2.8f * tile + 5.f) + (r4 % 2) * (2.f * tile + 5.f);
  const float groups = h > 1 ? r4 * (2.8f * half + 5.f) : INFINITY;  // the second group needs a grid row
  const float eight = r8 * (2.6f * tile + 5.f);
  if (four <= groups && four <= eight)
    return launch_f32_split<HD, CPR, 4, 1, 1>(q, kt, v, table, out, bh, h, w, scale, stream);
  if (groups <= eight) return launch_f32_split<HD, CPR, 4, 2, 1>(q, kt, v, table, out, bh, h, w, scale, stream);
  return launch_f32_split<HD, CPR, 8, 1, 2>(q, kt, v, table, out, bh, h, w, scale, stream);
}

template <int HD>
static hipError_t f32_split_cpr(const void* q, const void* kt, const void* v, const void* table, void* out, int bh,
                                int h, int w, float scale, hipStream_t stream) {
  switch ((w + 7) / 8) {
    case 1: return f32_split_waves<HD, 1>(q, kt, v, table, out, bh, h, w, scale, stream);
    case 2: return f32_split_waves<HD, 2>(q, kt, v, table, out, bh, h, w, scale, stream);
    case 3: return f32_split_waves<HD, 3>(q, kt, v, table, out, bh, h, w, scale, stream);
    case 4: return f32_split_waves<HD, 4>(q, kt, v, table, out, bh, h, w, scale, stream);
    case 5: return f32_split_waves<HD, 5>(q, kt, v, table, out, bh, h, w, scale, stream);
    case 6: return f32_split_waves<HD, 6>(q, kt, v, table, out, bh, h, w, scale, stream);
    case 7: return f32_split_waves<HD, 7>(q, kt, v, table, out, bh, h, w, scale, stream);
    default: return f32_split_waves<HD, 8>(q, kt, v, table, out, bh, h, w, scale, stream);
  }
}

// hd 64 and 80, grids up to 64 x 64; returns false (nothing launched) for other head dims and for more
// workgroups than a launch's 2^32 threads hold.
bool attn_relpos_f32_split(const void* q, const void* kt, const void* v, const void* table, void* out, int bh, int hd,
                           int h, int w, float scale, hipStream_t stream, hipError_t* err) {
  if ((hd != 64 && hd != 80) || h < 1 || h > 64 || w < 1 || w > 64) return false;
  if ((long)bh * ((h * w + 127) / 128) >= 1L << 23) return false;
  *err = hd == 64 ? f32_split_cpr<64>(q, kt, v, table, out, bh, h, w, scale, stream)
                  : f32_split_cpr<80>(q, kt, v, table, out, bh, h, w, scale, stream);
  return true;
}

}  // namespace samhip
