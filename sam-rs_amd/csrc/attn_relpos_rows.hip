// Fused rel-pos attention for grids of any size up to 64 x 63 at hd 64 and 80, f16 / bf16, for gfx950:
// the shapes that neither the 14x14 window kernel nor the 64-column kernel takes.
//
//   out[bh, r, :] = softmax_k( scale * q[r] . k[k] + q[r] . Th[i - kh + H-1] + q[r] . Tw[j - kw + W-1] ) . v
//
// The arithmetic and the operand layouts are those of attn_relpos.hip (S^T = K . Q^T with one query per
// lane, online exp2 softmax with a lazy rescale, O^T = V^T . P^T straight from the S^T accumulators).
// What differs is how the key grid is cut into tiles and how the work is spread:
//   * a grid row is padded to a multiple of 8 columns only (CPR chunks of 8) and the chunks of all rows
//     are packed one after the other into tiles of 64 slots. A 37 x 50 grid is 33 tiles instead of the 37
//     of one-row tiles, a 33-column grid 5/8 of them. A chunk is one (row, column group), and S^T block mb
//     gives lane half hh the columns 8 cc + 4 hh .. + 3 of its chunks 4 mb .. 4 mb + 3, so the Rw bias of
//     every column stays in 4 CPR registers for the whole loop; which chunk a tile starts with repeats
//     every CPR / gcd(CPR, 8) tiles, and the loop is unrolled by that, so that every register index is a
//     constant. The accumulators of a block start at (Rw + Rh) / scale, one add per score.
//   * kT rows are read by 16-byte loads at any 2-byte alignment (global loads take it), so that odd widths
//     cost no more than even ones.
//   * G = 2: the waves of a workgroup form two groups that take the upper and the lower half of the grid
//     rows for the same 128 queries and merge their (max, sum, O) through LDS at the end. A single image's
//     heads give too few 256-query blocks for the 256 CUs (16 heads of 37 x 50: 128 blocks); with 128
//     queries there are twice as many and each still has two waves per SIMD. G = 1 (4 waves, 128 queries)
//     serves grids of at most 128 tokens, whose halves would be a tile or less.
// What bounds it: like the 64-column kernel, the MFMA and the exp2 work of a SIMD's two waves.
#include <type_traits>

#include "lds_dma.hpp"
#include "relpos_geom.hpp"
#include "rows_tiles.hpp"

namespace samhip {

namespace rows {

constexpr float kSlack = 8.0f;
constexpr int kKStride = 64 + 16;  // elements of a kT row in LDS: transpose reads move 8 banks a row

template <int HD> struct Shape {
  static constexpr int kKS = HD / 16;
  static constexpr int kMBO = (HD + 31) / 32;
  static constexpr int kVStride = kMBO * 32 + 16;
  static constexpr bool kOnesRow = kMBO * 32 > HD;  // a spare O^T row carries the denominator
  static constexpr int kKBuf = HD * kKStride;       // elements
  static constexpr int kVBuf = 64 * kVStride;
  static constexpr int kTiles = 2 * (kKBuf + kVBuf);  // elements per wave group: two K and two V buffers
};

__device__ __forceinline__ int xcd_block(int i, int total) {
  const int per = total >> 3, rem = total & 7, x = i & 7, j = i >> 3;
  return x * per + (x < rem ? x : rem) + j;
}

typedef u32x4 __attribute__((aligned(2))) u32x4_a2;  // 16 bytes at any element

}  // namespace rows

template <typename T, int HD, int CPR, int NWV, int G>
__global__ __launch_bounds__(NWV * 64, 2) void attn_relpos_rows_kernel(
    const T* __restrict__ q, const T* __restrict__ kt, const T* __restrict__ v, const T* __restrict__ table,
    T* __restrict__ out, int H, int W, float scale, int qblocks) {
  using namespace rows;
  typedef Shape<HD> S;
  typedef typename Vec<T>::x8 X8;
  constexpr int kKS = S::kKS, kMBO = S::kMBO, kVStride = S::kVStride;
  constexpr bool kSplitP = __is_same(T, bf16);  // bf16: P as hi + lo for the P.V product
  constexpr int kQW = NWV / G;                  // query waves
  constexpr int kGT = kQW * 64;                 // threads of a group
  constexpr int kThreads = NWV * 64;
  constexpr int U = period(CPR);

  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qw = wave % kQW, grp = wave / kQW;
  const int gt = tid % kGT;
  T* kbase = reinterpret_cast<T*>(smem) + grp * S::kTiles;
  T* vbase = kbase + 2 * S::kKBuf;
  T* tbl = reinterpret_cast<T*>(smem);  // the table, during the prologue only
  const int R = H > W ? H : W;
  // per query wave: [row or column][query lane]; row R takes discarded scatters
  float* rhs = reinterpret_cast<float*>(reinterpret_cast<T*>(smem) + G * S::kTiles) + qw * (R + 1) * 32;

  const int N = H * W;
  const int n = lane & 31, hh = lane >> 5, g4 = lane >> 4, gi = lane & 15;
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  const long bh = blk / qblocks;
  const int q0 = (blk % qblocks) * (kQW * 32) + qw * 32;
  const bool active = q0 < N;  // whole wave
  const int qidx = q0 + n;
  const bool qvalid = qidx < N;
  const int qi = qvalid ? qidx / W : 0, qj = qvalid ? qidx % W : 0;

  // grid rows [r0, r1) of this group, and the tiles of the larger group (the first)
  const int hsplit = G == 1 ? H : (H + 1) / 2;
  const int r0 = grp == 0 ? 0 : hsplit, r1 = grp == 0 ? hsplit : H;
  const int ntiles = (hsplit * CPR + 7) / 8;

  // ---- staging: global -> registers -> LDS, with no masking in the steady state. Tile t starts at chunk
  // 8 t = (row 8 t / CPR, column group phase); a thread's chunk is a fixed distance from there, so its
  // offset is a few operations on constants of the phase, and the rest is a wave-uniform base.
  //   K: chunk gt % 8 of hd rows gt / 8 + u * kGT / 8. The columns of a row's last chunk past W are the next
  //   grid row's: real keys of this head, masked by the bias. Only in tiles with chunks that can reach past
  //   the head's end (first_end_row) are they cleared, and a load past that end starts earlier and is shifted.
  //   V: slot gt / kTPS, 16-byte pieces gt % kTPS + u * kTPS. Columns past W and rows past the group's are
  //   out of the buffer's range, which reads 0.
  constexpr int KPT = (HD * 8 + kGT - 1) / kGT;
  constexpr int kTPS = kGT / 64, VCPR = HD / 8, VPT = (VCPR + kTPS - 1) / kTPS;
  constexpr bool kKFull = HD * 8 % kGT == 0, kVFull = VCPR % kTPS == 0;
  u32x4 kreg[KPT], vreg[VPT];
  const T* ktb = kt + bh * HD * (long)N;
  const int kj = gt & 7, kd = gt >> 3;
  const int vsl = gt / kTPS, vpc = gt % kTPS;
  const bool kpart = kKFull || kd + (KPT - 1) * (kGT / 8) < HD;  // this thread's last K chunk exists (whole waves)
  const bool vpart = kVFull || vpc + (VPT - 1) * kTPS < VCPR;
  const int tailcols = W - 8 * (CPR - 1);  // 1..8 columns of a row's last chunk
  const bool vtail = (vsl & 7) < tailcols;
  const auto vrsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(v + (bh * N + r0 * W) * (long)HD), 0, (int)((r1 - r0) * W * HD * sizeof(T)), 0x00020000);
  // whether a K load of tile t can pass the head's end (either group's: the first reads on past its rows)
  const int first_end = first_end_row(H, W, CPR);
  auto has_end = [&](int t) { return reaches_row(t, r0, first_end, CPR); };
  auto k_x = [&](int t, auto uc) {
    constexpr int j0 = (8 * decltype(uc)::value) % CPR;
    return k_column(t, j0, (int)opaque(kj), r0, H, W, CPR);  // opaque: computed here, not held in a register per phase
  };
  auto load_k = [&](int t, auto uc) {
    const int x = k_x(t, uc);
    const bool end = has_end(t);
#pragma unroll
    for (int u = 0; u < KPT; ++u) {
      if (u + 1 < KPT || kpart) {
        unsigned off = (unsigned)(kd * N + x);
        if (end) off -= (unsigned)k_early(kd + u * (kGT / 8), x, N, HD);
        const char* base = reinterpret_cast<const char*>(ktb + (long)u * (kGT / 8) * N);
        kreg[u] = *reinterpret_cast<const u32x4_a2*>(base + off * (unsigned)sizeof(T));
      }
    }
  };
  auto load_v = [&](int t, auto uc) {
    constexpr int j0 = (8 * decltype(uc)::value) % CPR;
    const int sl = (int)opaque(vsl);
    const int j = j0 + (sl >> 3), add = j / CPR, cc = j - add * CPR;
    const bool ok = cc < CPR - 1 || vtail;
    const int off = ok ? (int)(((add * W + 8 * cc + (sl & 7)) * HD + 8 * vpc) * sizeof(T)) : 0x40000000;
    const int base = (int)(v_row(t, r1 - r0, CPR) * W * HD * sizeof(T));
#pragma unroll
    for (int u = 0; u < VPT; ++u)
      if (u + 1 < VPT || vpart)
        vreg[u] = __builtin_amdgcn_raw_buffer_load_b128(vrsrc, off + 16 * kTPS * u, base, 0);
  };
  auto store_k = [&](int t, auto uc) {
    T* kbuf = kbase + (t & 1) * S::kKBuf + kd * kKStride + 8 * kj;
    if (has_end(t)) {
      constexpr int j0 = (8 * decltype(uc)::value) % CPR;
      const int x = k_x(t, uc);
      const bool tail = (j0 + kj) % CPR == CPR - 1;
#pragma unroll
      for (int u = 0; u < KPT; ++u) {
        const int early = k_early(kd + u * (kGT / 8), x, N, HD);
        if (wave_any(early > 0)) {
          const unsigned long lo = ((unsigned long)kreg[u][1] << 32) | kreg[u][0];
          const unsigned long hi = ((unsigned long)kreg[u][3] << 32) | kreg[u][2];
          const int sh = 16 * (early & 3);
          const unsigned long a = early & 4 ? hi : lo, b = early & 4 ? 0 : hi;
          const unsigned long y = (a >> sh) | (sh ? b << (64 - sh) : 0), z = b >> sh;
          kreg[u] = u32x4{(unsigned)y, (unsigned)(y >> 32), (unsigned)z, (unsigned)(z >> 32)};
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const unsigned m = tailcols >= 2 * i + 2 ? 0xffffffffu : (tailcols == 2 * i + 1 ? 0xffffu : 0u);
          kreg[u][i] = tail ? kreg[u][i] & m : kreg[u][i];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < KPT; ++u)
      if (u + 1 < KPT || kpart) *reinterpret_cast<u32x4*>(kbuf + u * (kGT / 8) * kKStride) = kreg[u];
  };
  auto store_v = [&](int t) {
    T* vbuf = vbase + (t & 1) * S::kVBuf + vsl * kVStride + 8 * vpc;
#pragma unroll
    for (int u = 0; u < VPT; ++u)
      if (u + 1 < VPT || vpart) *reinterpret_cast<u32x4*>(vbuf + 8 * kTPS * u) = vreg[u];
  };

  // ---- prologue: first tiles in flight, q fragments, the table into LDS
  X8 qf[kKS];
  {
    const T* qrow = q + (bh * N + (qvalid ? qidx : 0)) * HD;
#pragma unroll
    for (int s = 0; s < kKS; ++s) qf[s] = *reinterpret_cast<const X8*>(qrow + 16 * s + 8 * hh);
  }
  const int trows = 2 * H - 1 + 2 * W - 1;
  for (int c = tid; c < trows * (HD / 8); c += kThreads)
    *reinterpret_cast<u32x4*>(tbl + c * 8) = *reinterpret_cast<const u32x4*>(table + c * 8);
  typedef std::integral_constant<int, 0> P0;
  load_k(0, P0());
  load_v(0, P0());
  __syncthreads();

  // Rw and Rh bands, G = T . Q^T on the MFMA in 32-row blocks, scattered along the diagonal, divided by
  // the scale (the MFMA accumulators start from them). Entries outside the band go to the junk row.
  const float rscale = 1.f / scale;
  auto band = [&](const T* tab, int nrows, int base, int len, auto maxb) {
#pragma unroll
    for (int b = 0; b < decltype(maxb)::value; ++b) {
      if (32 * b < nrows) {
        f32x16 acc = {};
#pragma unroll
        for (int s = 0; s < kKS; ++s) {
          // rows past the end of a table hold other rows or stale data and are never scattered
          const X8 a = *reinterpret_cast<const X8*>(tab + (32 * b + n) * HD + 16 * s + 8 * hh);
          acc = mma32(a, qf[s], acc);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int rr = 32 * b + 8 * (e >> 2) + 4 * hh + (e & 3);
          const int k = base + len - 1 - rr;  // kh = i + H-1 - rr, kw = j + W-1 - rr
          const bool ok = rr < nrows && k >= 0 && k < len;
          rhs[(ok ? k : R) * 32 + n] = acc[e] * rscale;
        }
      }
    }
  };
  if (active && grp == 0)
    band(tbl + (2 * H - 1) * HD, 2 * W - 1, qj, W, std::integral_constant<int, (16 * CPR - 1 + 31) / 32>());
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
  if (active && grp == G - 1) band(tbl, 2 * H - 1, qi, H, std::integral_constant<int, 4>());
  __syncthreads();  // the table region is free from here on

  store_k(0, P0());
  store_v(0);
  for (int i = gt; i < 2 * 64; i += kGT) {
    T* rowp = vbase + (i >> 6) * S::kVBuf + (i & 63) * kVStride;
    for (int c = HD; c < kVStride; ++c) rowp[c] = from_f32<T>((S::kOnesRow && c == HD) ? 1.f : 0.f);
  }
  __syncthreads();

  // per-lane addresses of the transpose reads; tiles, k-steps and blocks are constants added to them
  const T* kl = kbase + (8 * (g4 >> 1) + (gi >> 2)) * kKStride + 16 * (g4 & 1) + 4 * (gi & 3);
  const T* vl = vbase + (4 * (g4 >> 1) + (gi >> 2)) * kVStride + 16 * (g4 & 1) + 4 * (gi & 3);

  const float sc = scale * kLog2e;
  // The maximum starts at a finite value: infinite keys can make all of a query's scores in a group's tiles so far
  // -inf, and those must weigh 0. (A test for it in the loop takes a register and two instructions a tile.)
  float m_run = -3e38f, l_run = 0.f;
  f32x16 o[kMBO];
#pragma unroll
  for (int ob = 0; ob < kMBO; ++ob) o[ob] = f32x16{};

  // S^T of tile t (pattern phase uc = t % U), bias included; rows past the group's are masked by it
  auto qk = [&](int t, auto uc, f32x16* s) {
    constexpr int j0 = (8 * decltype(uc)::value) % CPR;
    const int row0 = r0 + (8 * t) / CPR;
    const T* kp = kl + (t & 1) * S::kKBuf;
    float rh[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j == 0 || (j0 + j) % CPR == 0) {
        const int row = row0 + (j0 + j) / CPR;
        const float x = rhs[(row < r1 ? row : r0) * 32 + n];
        rh[j] = row < r1 ? x : -INFINITY;
      } else {
        rh[j] = rh[j - 1];
      }
    }
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        s[mb][e] = rw[4 * ((j0 + 4 * mb + (e >> 2)) % CPR) + (e & 3)] + rh[4 * mb + (e >> 2)];
#pragma unroll
      for (int k = 0; k < kKS; ++k) {
        const T* p = kp + 32 * mb + 16 * k * kKStride;
        s[mb] = mma32(join8<T>(lds_read_tr16(p), lds_read_tr16(p + 4 * kKStride)), qf[k], s[mb]);
      }
    }
  };

  // One tile: the next one's loads, S^T, softmax, P.V. Issuing the next tile's S^T ahead of the softmax, as
  // the one-tile-a-row kernels do, was 1-4% slower here: its 32 registers push the hd 80 kernel into
  // spills, and the two waves of a SIMD already overlap.
  auto step = [&](int t, auto uc) {
    typedef std::integral_constant<int, (decltype(uc)::value + 1) % U> Next;
    load_k(t + 1, Next());
    load_v(t + 1, Next());
    if (active) {
      f32x16 s_cur[2];
      qk(t, uc, s_cur);
      float mm = s_cur[0][0];
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int e = 0; e < 16; ++e) mm = max_nc(mm, s_cur[mb][e]);
      const float mt = max_with_partner32(mm * sc);
      if (wave_any(mt > m_run + kSlack)) {
        const float m_new = fmaxf(m_run, mt);
        const float alpha = exp2_fast(m_run - m_new);
        l_run *= alpha;
#pragma unroll
        for (int ob = 0; ob < kMBO; ++ob) o[ob] *= alpha;
        m_run = m_new;
      }
      X8 b[4], blo[4];
#pragma unroll
      for (int w4 = 0; w4 < 4; ++w4) {
        float pv[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) pv[e] = exp2_fast(fmaf(s_cur[w4 >> 1][8 * (w4 & 1) + e], sc, -m_run));
        if constexpr (kSplitP)
          split_hi_lo(pv, b[w4], blo[w4]);
        else
          b[w4] = pack8(pv, (X8*)nullptr);
        if constexpr (!S::kOnesRow) {
          if constexpr (!kSplitP) {
            // f16: the sum over P as the P.V product sees it (rounded)
            typedef _Float16 h2 __attribute__((ext_vector_type(2)));
#pragma unroll
            for (int e = 0; e < 8; e += 2)
              l_run = __builtin_amdgcn_fdot2(h2{b[w4][e], b[w4][e + 1]}, h2{(f16)1.f, (f16)1.f}, l_run, false);
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) l_run += pv[e];
          }
        }
      }
      const T* vp = vl + (t & 1) * S::kVBuf;
#pragma unroll
      for (int w4 = 0; w4 < 4; ++w4)
#pragma unroll
        for (int ob = 0; ob < kMBO; ++ob) {
          const T* p = vp + 16 * w4 * kVStride + 32 * ob;
          const X8 a = join8<T>(lds_read_tr16(p), lds_read_tr16(p + 8 * kVStride));
          o[ob] = mma32(a, b[w4], o[ob]);
          if (kSplitP) o[ob] = mma32(a, blo[w4], o[ob]);
        }
    }
    store_k(t + 1, Next());  // over tile t - 1, which every wave left before the last barrier
    store_v(t + 1);
    __syncthreads();
  };

  for (int t = 0; t < ntiles; t += U) {
    step(t, P0());
#define SAMHIP_ROWS_STEP(i) \
  if constexpr ((i) < U)    \
    if (t + (i) < ntiles) step(t + (i), std::integral_constant<int, (i) % U>());
    SAMHIP_ROWS_STEP(1)
    SAMHIP_ROWS_STEP(2)
    SAMHIP_ROWS_STEP(3)
    SAMHIP_ROWS_STEP(4)
    SAMHIP_ROWS_STEP(5)
    SAMHIP_ROWS_STEP(6)
#undef SAMHIP_ROWS_STEP
  }

  // ---- the denominator of this group's keys, the same in both lanes of a query
  float l;
  if constexpr (S::kOnesRow) {
    // O^T row HD (= 32 (MBO - 1) + 16): element 8 of the lower lane half
    const unsigned x = __float_as_uint(o[kMBO - 1][8]);
    auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    l = __uint_as_float(r[0]);
  } else {
    l = sum_with_partner32(l_run);
  }
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
  if (qvalid) {
    T* orow = out + (bh * N + qidx) * HD;
#pragma unroll
    for (int ob = 0; ob < kMBO; ++ob)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        if (32 * ob + 8 * a < HD) {
          typename Vec<T>::x4 w4;
#pragma unroll
          for (int bb = 0; bb < 4; ++bb) w4[bb] = from_f32<T>(o[ob][4 * a + bb] * inv);
          *reinterpret_cast<typename Vec<T>::x4*>(orow + 32 * ob + 8 * a + 4 * hh) = w4;
        }
      }
  }
}

template <typename T, int HD, int CPR, int NWV, int G>
static hipError_t launch_rows(const void* q, const void* kt, const void* v, const void* table, void* out, int bh,
                              int h, int w, float scale, hipStream_t stream) {
  typedef rows::Shape<HD> S;
  constexpr int kQW = NWV / G;
  constexpr size_t tiles = (size_t)G * S::kTiles * sizeof(T);
  static_assert(tiles + kQW * 65 * 32 * sizeof(float) <= 160 * 1024, "LDS");
  static_assert(254 * HD * sizeof(T) <= tiles, "the table must fit in the tile buffers during the prologue");
  static_assert(G == 1 || kQW * (16 * S::kMBO + 2) * 64 * sizeof(float) <= tiles, "the exchange must fit there too");
  auto kern = attn_relpos_rows_kernel<T, HD, CPR, NWV, G>;
  static std::atomic<unsigned long long> lds_done{0};
  if (const hipError_t e = lds_opt_in(lds_done, (const void*)kern, (int)(tiles + kQW * 65 * 32 * sizeof(float)));
      e != hipSuccess)
    return e;
  const int r = h > w ? h : w;
  const size_t lds = tiles + (size_t)kQW * (r + 1) * 32 * sizeof(float);
  const int qblocks = (h * w + kQW * 32 - 1) / (kQW * 32);
  hipLaunchKernelGGL(kern, dim3((unsigned)(bh * qblocks)), dim3(NWV * 64), lds, stream, (const T*)q, (const T*)kt,
                     (const T*)v, (const T*)table, (T*)out, h, w, scale, qblocks);
  return hipGetLastError();
}

// Whether two wave groups of 128 queries beat one of 256. A workgroup has a CU to itself (8 waves of over 128
// registers), so the time is that of the fullest CU: rounds of workgroups times (key tiles per wave + the
// prologue and epilogue, about 5 tiles' time). A tile costs a group of the split form 1.2 times as much,
// since its 4 waves stage it alone. Measured at hd 80, f16, split against one group: 16 heads of 37 x 50
// 41.9 / 64.0 us, 24 of 32 x 32 22.9 / 32.7, 64 of 15 x 15 11.5 / 12.9, 192 of 24 x 24 64.7 / 60.0, 160 of
// 12 x 12 20.0 / 11.4.
static bool rows_split(int bh, int h, int w) {
  const int cus = device_cu_count(), n = h * w, cpr = (w + 7) / 8;
  const long b1 = (long)bh * ((n + 255) / 256), b2 = (long)bh * ((n + 127) / 128);
  const long r1 = (b1 + cus - 1) / cus, r2 = (b2 + cus - 1) / cus;
  const float t1 = (float)((h * cpr + 7) / 8), t2 = (float)(((h + 1) / 2 * cpr + 7) / 8);
  return r2 * (1.2f * t2 + 5.f) < r1 * (t1 + 5.f);
}

template <typename T, int HD, int CPR>
static hipError_t pick_waves(const void* q, const void* kt, const void* v, const void* table, void* out, int bh, int h,
                             int w, float scale, hipStream_t stream) {
  if (h * w <= 128) return launch_rows<T, HD, CPR, 4, 1>(q, kt, v, table, out, bh, h, w, scale, stream);
  if (rows_split(bh, h, w)) return launch_rows<T, HD, CPR, 8, 2>(q, kt, v, table, out, bh, h, w, scale, stream);
  return launch_rows<T, HD, CPR, 8, 1>(q, kt, v, table, out, bh, h, w, scale, stream);
}

template <typename T, int HD>
static hipError_t pick_cpr(const void* q, const void* kt, const void* v, const void* table, void* out, int bh, int h,
                           int w, float scale, hipStream_t stream) {
  switch ((w + 7) / 8) {
    case 1: return pick_waves<T, HD, 1>(q, kt, v, table, out, bh, h, w, scale, stream);
    case 2: return pick_waves<T, HD, 2>(q, kt, v, table, out, bh, h, w, scale, stream);
    case 3: return pick_waves<T, HD, 3>(q, kt, v, table, out, bh, h, w, scale, stream);
    case 4: return pick_waves<T, HD, 4>(q, kt, v, table, out, bh, h, w, scale, stream);
    case 5: return pick_waves<T, HD, 5>(q, kt, v, table, out, bh, h, w, scale, stream);
    case 6: return pick_waves<T, HD, 6>(q, kt, v, table, out, bh, h, w, scale, stream);
    case 7: return pick_waves<T, HD, 7>(q, kt, v, table, out, bh, h, w, scale, stream);
    default: return pick_waves<T, HD, 8>(q, kt, v, table, out, bh, h, w, scale, stream);
  }
}

// Grids of up to 64 x 64 at hd 64 and 80 for scales of ordinary size (the accumulators start at the bias
// divided by the scale, as in the 64-column kernel); returns false (nothing launched) for other shapes.
// Widths of 25..32 and 57..64 pack no better than the general kernel's tiles of two or one whole rows. Its
// steps are a little shorter there when the width is even, so it keeps what is not split, except at hd 64
// past one round of workgroups (bf16, this kernel against it: 43 heads of 33 x 58 131 / 135 us, 60 of 60 x 58
// 448 / 459), and in f16 only where two of this kernel's workgroups share a CU, their registers (25..32 columns)
// and their bias scratch of max(h, w) rows both fitting: 273 heads of 27 x 32 115 / 142, 152 of 32 x 26 78 / 96, but
// 146 of 52 x 32 196 / 182, and of one workgroup a CU 69 of 56 x 62 382 / 368. Odd widths gain (bf16 59 x 63
// 132 / 214).
bool attn_relpos_rows(int dtype, const void* q, const void* kt, const void* v, const void* table, void* out, int bh,
                      int hd, int h, int w, float scale, hipStream_t stream, hipError_t* err) {
  const float sc = scale * kLog2e;
  if ((hd != 80 && hd != 64) || h < 1 || h > 64 || w < 1 || w > 64 || !(sc >= 0.015625f && sc <= 4.f)) return false;
  const int cpr = (w + 7) / 8;
  if ((cpr == 4 || cpr == 8) && w % 2 == 0 && h * w > 128 && !rows_split(bh, h, w)) {
    const bool one_round = (long)bh * ((h * w + 255) / 256) <= device_cu_count();
    const size_t lds = rows::Shape<64>::kTiles * sizeof(f16) + (size_t)8 * ((h > w ? h : w) + 1) * 32 * sizeof(float);
    const bool two_a_cu = cpr == 4 && 2 * lds <= 160 * 1024;
    if (hd == 80 || one_round || (dtype == kF16 && !two_a_cu)) return false;
  }
  if (hd == 80)
    *err = dtype == kF16 ? pick_cpr<f16, 80>(q, kt, v, table, out, bh, h, w, scale, stream)
                         : pick_cpr<bf16, 80>(q, kt, v, table, out, bh, h, w, scale, stream);
  else
    *err = dtype == kF16 ? pick_cpr<f16, 64>(q, kt, v, table, out, bh, h, w, scale, stream)
                         : pick_cpr<bf16, 64>(q, kt, v, table, out, bh, h, w, scale, stream);
  return true;
}

}  // namespace samhip
