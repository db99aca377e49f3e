// The batched prefill's exact projections (B256, prefill.h) on the matrix
// cores.
//
// v_mfma_f32_16x16x4_f32 adds its four products to the accumulator one after
// another, k = 0 .. 3, each as a fused multiply-add rounded once (checked on
// the device against chains of fmaf: signs, subnormals, cancellation). A
// product of two BF16 values is exact in F32 as long as it neither underflows
// nor overflows, and then fma(x, w, acc) is acc + x * w rounded separately:
// the reference's B256 lane step, bit for bit. So one instruction runs two
// visits (lo, hi, lo, hi) of one reference lane for a 16 x 16 tile of
// outputs; the lanes' 256-wide halving tree stays on the vector unit. A
// padded visit adds 0 * 0, which leaves a chain that began at +0 as it is.
//
// Products outside that range: the block of a row tile's first token tile
// reads the smallest non-zero and the largest magnitude of its weights (which
// it is about to stage), the block of the first row tile those of its token
// tile, and k_bgemm_fix, launched
// behind, recomputes every output tile whose products may leave the range in
// the separate-rounding order (normally none).
//
// Split. A wave of the block's eight owns quad c (16 bytes, reference lanes
// 4c .. 4c+3) of every 128-byte line of K, so the block consumes whole lines:
// line 8 s + L holds visit s of the lanes 32 L .. 32 L + 31. For each L the
// wave runs the four lanes' chains over s, and the lines are taken in the
// order 0 4 2 6 1 5 3 7 so that the tree's strides 128, 64 and 32 become
// register adds of at most three live levels (the first half's sum waits in
// LDS). Strides 16, 8, 4 (the waves) and 2, 1 (in the quad) are added at the
// end, one output per thread, through LDS. Two visits of all rows are staged
// per barrier with whole-line loads straight into LDS, three stages ahead.
//
// Bound: no one unit. The F32 matrix instructions alone run at 75 T
// multiply-adds/s on this part; 12352 rows x 2048 columns x 768 tokens take 653
// us, 29.8 T/s, 2048 x 6144 279 us, 34.7 T/s. Counters of the plain 48 x 16
// form (2B layers, 777 tokens): the matrix cores are busy 40 % of a SIMD's
// cycles (46 % in the residual form), other vector instructions (4.4 per
// matrix instruction: operands, tree adds, addresses) issue in 22 %, and for
// the rest neither: a SIMD's two waves are in the same stage, with a barrier
// per 12 matrix instructions, and spend 27 % of their time in waits and 44 %
// with an instruction ready that the unit is not free for. LDS is active 22 %
// of the time, three tenths of that conflicts; with all loads
// taken out the kernel is 8 % faster. Wider tiles (48 x 16 is what the
// registers hold: 64 sums of three levels) gain little. The vector kernel
// (k_bproject) reached 11 T/s: eight 2B layers of a 777-token prompt went from
// 43.4 to 20.4 ms.
#pragma once

#include "prefill.h"

namespace cq35 {

constexpr int kEWaves = 8;
constexpr int kEThreads = 64 * kEWaves;

// Token tiles of 16 per block, by one of 16 weight rows.
template <int TT>
struct BGemmTile {
  static constexpr int kTokens = 16 * TT, kRows = 16, kStaged = kTokens + kRows;
  static constexpr int kOut = 256 * TT;            // outputs per block
  static constexpr int kStage = kStaged * 16;      // 16-byte pieces per stage (two lines per row)
  static constexpr int kLoads = (kStage + kEThreads - 1) / kEThreads;
  // the waves' sums: 4 lanes of the quad x kOut F32 each
  static constexpr size_t kSums = (size_t)kEWaves * 4 * kOut * 4;
  static constexpr int kBufs = 4;  // LDS stages: one read, the others on their way
  static constexpr size_t kLds = kSums + kBufs * (size_t)kStage * 16;
  static constexpr int kBlocksPerCu = TT == 1 ? 2 : 1;
};

// What a piece past the end of a row reads.
__device__ const u32x4 bg_zeros[1] = {{0u, 0u, 0u, 0u}};

// Smallest non-zero and largest BF16 magnitude (15 bits each) of the words a
// thread has seen, two values at a time.
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
struct BfRange {
  u16x2 low = {0xffff, 0xffff}, high = {0, 0};  // 2 m - 1 (zero: 65535), 2 m
  __device__ __forceinline__ void add(uint32_t w) {
    const u16x2 v = __builtin_bit_cast(u16x2, w) * (uint16_t)2;  // drops the sign
    low = __builtin_elementwise_min(low, (u16x2)(v - (uint16_t)1));
    high = __builtin_elementwise_max(high, v);
  }
  __device__ __forceinline__ void add(const u32x4& q) {
    add(q.x);
    add(q.y);
    add(q.z);
    add(q.w);
  }
};

// A tile's range as one word: smallest non-zero 2 m - 1 above, largest 2 m
// below. Whether every product of a token tile's and a weight tile's values
// is exact in F32: its lowest bit at or above 2^-149, its magnitude below
// 2^128, nothing infinite or NaN.
__device__ __forceinline__ bool bf_products_exact(uint32_t x, uint32_t w) {
  auto lowest = [](uint32_t r) {  // exponent of the lowest bit of the smallest non-zero value
    const int e = (int)((r >> 16) >> 8);
    return e > 0 ? e - 134 : -133;
  };
  auto highest = [](uint32_t r) { return (int)((r & 0xffffu) >> 8) - 126; };  // all magnitudes below 2^this
  if ((x >> 16) == 0xffffu || (w >> 16) == 0xffffu) return ((x & 0xffffu) >> 8) < 255u && ((w & 0xffffu) >> 8) < 255u;
  return lowest(x) + lowest(w) >= -149 && highest(x) + highest(w) <= 128 && highest(x) < 129 && highest(w) < 129;
}

// A tile's range over its kEWaves words.
__device__ __forceinline__ uint32_t range_of(const uint32_t* ranges, int tile) {
  const u32x4* p = reinterpret_cast<const u32x4*>(ranges + (size_t)tile * kEWaves);
  uint32_t low = 0xffffu, high = 0;
#pragma unroll
  for (int k = 0; k < kEWaves / 4; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      low = min(low, p[k][i] >> 16);
      high = max(high, p[k][i] & 0xffffu);
    }
  return low << 16 | high;
}

// Output rows per block: in gate mode a tile holds eight gate rows and the
// same eight up rows.
template <int kMode>
constexpr int bgemm_rows() { return kMode == kBGate ? 8 : 16; }

// out_s[t][r] of n token rows against the concatenated rows of `seg` (gate
// mode: one segment, w2 the up matrix), k_bproject's epilogues. cols % 64 ==
// 0. One block per CU walks its tiles, the next tile's first stage requested
// before the current one's last sums. Block b runs on XCD b mod 8 and takes
// row tiles = b mod 8: a row tile's token tiles follow each other there, so a
// weight tile comes from HBM once. `ranges`: kEWaves words per row tile, then
// per token tile.
template <int kMode, int TT>
__global__ __launch_bounds__(kEThreads, (2 * BGemmTile<TT>::kBlocksPerCu)) void k_bgemm(const uint16_t* __restrict__ x, int n, int cols, Segments seg,
                                                     const uint16_t* __restrict__ w2,
                                                     const uint16_t* __restrict__ res,
                                                     uint32_t* __restrict__ ranges) {
  using T = BGemmTile<TT>;
  constexpr int kBlockRows = bgemm_rows<kMode>();
  extern __shared__ __align__(16) u32x4 bg_lds[];
  f32x4* sums = reinterpret_cast<f32x4*>(bg_lds);
  u32x4* stage = bg_lds + T::kSums / 16;
  const int rows = seg.rows[0] + seg.rows[1] + seg.rows[2] + seg.rows[3];
  const int tiles_t = (n + T::kTokens - 1) / T::kTokens, tiles_r = (rows + kBlockRows - 1) / kBlockRows;
  const int xcd = blockIdx.x & 7, step = gridDim.x >> 3;
  const int count = ((tiles_r - xcd + 7) >> 3) * tiles_t;  // this XCD's tiles
  int at = blockIdx.x >> 3;                                // the current one
  if (at >= count) return;
  const int lane = threadIdx.x & 63, c = threadIdx.x >> 6;
  const int lines = cols >> 6;          // 128-byte lines per row
  const int pairs = (lines + 15) >> 4;  // stages per L: two visits of 512 columns each
  // the lines in an order of the block's own (the tree's pairs are the same
  // for L ^ turn), so that the CUs do not all ask the same cache channels
  const int turn = at & 7;

  // this thread's pieces of a stage: row (tokens, then weights), visit of the
  // pair, piece of the line
  const uint16_t* src[T::kLoads];
  // the thread index behind a fence: what is computed from it is not held in
  // registers across the chains
  auto tid_here = [&]() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
  };
  auto aim = [&](int tile) {
    const int tid = tid_here();
    const int t0 = (tile % tiles_t) * T::kTokens, r0 = ((tile / tiles_t) * 8 + xcd) * kBlockRows;
#pragma unroll
    for (int k = 0; k < T::kLoads; ++k) {
      const int i = min(tid + kEThreads * k, T::kStage - 1);
      const int row = i >> 4, visit = (i >> 3) & 1, piece = i & 7;
      const uint16_t* base;
      if (row < T::kTokens) {
        base = x + (size_t)min(t0 + row, n - 1) * cols;
      } else {
        int wr = row - T::kTokens;
        const bool up = kMode == kBGate && (wr & 8) != 0;
        if (kMode == kBGate) wr &= 7;
        int local;
        const int s = segment_of(seg, min(r0 + wr, rows - 1), &local);
        base = (up ? w2 : segment_w(seg, s)) + (size_t)local * cols;
      }
      src[k] = base + 512 * visit + 8 * (piece ^ (row & 7));
    }
  };
  // A stage goes straight into LDS (16 bytes per lane, no registers held):
  // slot i of a buffer holds row i / 16, visit (i / 8) % 2, piece (i % 8) ^
  // (row % 8), so that the 16 rows of an operand read spread over the banks.
  // The stage behind the last requested one: line f_line of the order below,
  // visit pair f_sp, of tile f_at; `src` points into that tile.
  const uint32_t wave_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) u32x4*)stage +
                            1024u * (uint32_t)__builtin_amdgcn_readfirstlane(c);
  int f_at = at, f_line = 0, f_sp = 0, f_buf = 0;
  auto line_at = [&](int i) { return (int)(0x73516240u >> (4 * i) & 7u) ^ turn; };
  auto fetch = [&]() {
    if (f_at >= count) return;
    const int line = 16 * f_sp + line_at(f_line);
    const bool whole = line + 8 < lines;  // uniform: both visits inside the row
#pragma unroll
    for (int k = 0; k < T::kLoads; ++k) {
      const uint16_t* from = src[k] + 64 * line;
      if (!whole && line + (tid_here() & 8) >= lines) from = reinterpret_cast<const uint16_t*>(bg_zeros);  // visit 1 adds eight lines
      // 16 bytes per lane to LDS (M0: the wave's place); written out because
      // the compiler would make every later LDS read wait for all of them
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                   :
                   : "s"(wave_lds + 16u * (uint32_t)(f_buf * T::kStage + kEThreads * k)), "v"(from)
                   : "memory", "m0");
    }
    f_buf = f_buf + 1 == T::kBufs ? 0 : f_buf + 1;
    if (++f_sp == pairs) {
      f_sp = 0;
      if (++f_line == 8) {
        f_line = 0;
        f_at += step;
        if (f_at < count) aim(f_at);
      }
    }
  };
  // The next stage is in LDS, for every wave. Requests complete in their
  // order, so the newer stages' may stay outstanding (stores among them make
  // the wait longer, never shorter); behind the last request, none.
  auto arrived = [&]() {
    __builtin_amdgcn_sched_barrier(0);  // no operands of this stage held past it but lane j = 3's
    if (f_at >= count) __builtin_amdgcn_s_waitcnt(0x0f70);               // vmcnt(0)
    else __builtin_amdgcn_s_waitcnt(0x0f70 | (T::kBufs - 2) * T::kLoads);  // vmcnt(requests of the newer stages)
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
  };
  // The range of m rows from row0 of x (weights: of the launch's rows), one
  // word per wave into `to`. Ahead of a tile's chains, when no sums are held.
  auto note = [&](bool weights, int row0, int m, uint32_t* to) {
    BfRange g;
    const int quads = cols >> 3;
    for (int row = c; row < m; row += kEWaves) {
      const uint16_t* base;
      if (weights) {
        const bool up = kMode == kBGate && (row & 8) != 0;
        int local;
        const int s = segment_of(seg, min(row0 + (kMode == kBGate ? row & 7 : row), rows - 1), &local);
        base = (up ? w2 : segment_w(seg, s)) + (size_t)local * cols;
      } else {
        base = x + (size_t)min(row0 + row, n - 1) * cols;
      }
#pragma unroll 4
      for (int q = lane; q < quads; q += 64) g.add(ldq(base, q));
    }
    uint32_t v = (uint32_t)min(g.low.x, g.low.y) << 16 | max(g.high.x, g.high.y);
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
      const uint32_t o = __shfl_xor(v, d, 64);
      v = min(v >> 16, o >> 16) << 16 | max(v & 0xffffu, o & 0xffffu);
    }
    if (lane == 0) to[c] = v;
  };

  // operand lane l: row l % 16 of a tile, k = l / 16: visit k / 2, low or
  // high half of the pair. A stage's lane j = 3 is multiplied behind the next
  // stage's LDS reads, whose latency it covers.
  const int i16 = lane & 15, visit = lane >> 5;
  const uint32_t half = (lane >> 4) & 1 ? 0x03020c0cu : 0x01000c0cu;
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 a0[4][TT], a1[4][TT], a2[4][TT];  // lines' sums
  u32x4 a[TT], b;
  float a3[TT], b3;
  auto read = [&](int buf) {
    const u32x4* s = stage + buf * T::kStage;
    auto piece = [&](int row) { return s[(row * 2 + visit) * 8 + (c ^ (row & 7))]; };
#pragma unroll
    for (int t = 0; t < TT; ++t) a[t] = piece(16 * t + i16);
    b = piece(T::kTokens + i16);
  };
  auto multiply = [&](f32x4 (&acc)[4][TT], auto first) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float af[TT];
#pragma unroll
      for (int t = 0; t < TT; ++t) af[t] = bitsf(__builtin_amdgcn_perm(0u, a[t][j], half));
      const float bf = bitsf(__builtin_amdgcn_perm(0u, b[j], half));
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        if (j == 3) a3[t] = af[t];
        else acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[t], bf, decltype(first)::value ? zero : acc[j][t], 0, 0, 0);
      }
      if (j == 3) b3 = bf;
    }
  };
  auto last_lane = [&](f32x4 (&acc)[4][TT], auto first) {
#pragma unroll
    for (int t = 0; t < TT; ++t)
      acc[3][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a3[t], b3, decltype(first)::value ? zero : acc[3][t], 0, 0, 0);
  };

  static_assert(T::kStage % kEThreads == 0 && T::kBufs >= 2, "requests per stage");
  aim(at);
  int buf = 0;
#pragma unroll 1
  for (int i = 0; i < T::kBufs - 1; ++i) fetch();
  arrived();
  f32x4* mine = sums + (size_t)c * 4 * TT * 64;  // [j][tile][lane]
  // what becomes of the sums when a line is done, lanes j0 .. j1 - 1: a half's
  // lines 0 and 1 go to a0 and a1 (a0 += a1), 2 and 3 to a1 and a2
  auto fold = [&](auto k, int j0, int j1) {
#pragma unroll
    for (int j = j0; j < j1; ++j)
#pragma unroll
      for (int i = 0; i < TT; ++i) {
        f32x4* m = &mine[(j * TT + i) * 64 + lane];
        if (k() == 1) a0[j][i] = a0[j][i] + a1[j][i];
        if (k() == 3) *m = a0[j][i] + (a1[j][i] + a2[j][i]);
        if (k() == 4) *m = *m + (a0[j][i] + (a1[j][i] + a2[j][i]));
      }
  };
  // the last products of line k of a half (4: of the second half's line 3)
  auto finish_line = [&](auto k) {
    f32x4(&acc)[4][TT] = k() == 0 ? a0 : k() < 3 ? a1 : a2;
    fold(k, 0, 3);
    if (pairs == 1) last_lane(acc, std::true_type{});
    else last_lane(acc, std::false_type{});
    fold(k, 3, 4);
  };
  while (true) {
    const int tile_t = at % tiles_t, tile_r = (at / tiles_t) * 8 + xcd;
    const int t0 = tile_t * T::kTokens, r0 = tile_r * kBlockRows;
    // (a block's tiles are all of one token tile where tiles_t divides the
    // step, so the noting one moves with the row tile)
    if (tile_t == (tile_r >> 3) % tiles_t) note(true, r0, T::kRows, ranges + (size_t)tile_r * kEWaves);
    if (tile_r == tile_t % tiles_r) note(false, t0, T::kTokens, ranges + (size_t)(tiles_r + tile_t) * kEWaves);
    // lines 0 4 2 6, then 1 5 3 7 (each ^ turn)
#pragma unroll 1
    for (int h = 0; h < 2; ++h) {
      // line k's chains
      auto run_line = [&](auto k) {
        f32x4(&acc)[4][TT] = k() == 0 ? a0 : k() < 3 ? a1 : a2;
        auto one = [&](int sp, auto first) {
          if (decltype(first)::value) {
            if (k() != 0) finish_line(std::integral_constant<int, (decltype(k)::value + 3) % 4>{});
            else if (h == 1) finish_line(std::integral_constant<int, 3>{});
          }
          __builtin_amdgcn_sched_barrier(0);
          read(buf);
          if (!decltype(first)::value) {
            if (sp == 1) last_lane(acc, std::true_type{});
            else last_lane(acc, std::false_type{});
          }
          fetch();
          multiply(acc, first);
          arrived();
          buf = buf + 1 == T::kBufs ? 0 : buf + 1;
        };
        one(0, std::true_type{});
#pragma unroll 1
        for (int sp = 1; sp < pairs; ++sp) one(sp, std::false_type{});
      };
      run_line(std::integral_constant<int, 0>{});
      run_line(std::integral_constant<int, 1>{});
      run_line(std::integral_constant<int, 2>{});
      run_line(std::integral_constant<int, 3>{});
    }
    finish_line(std::integral_constant<int, 4>{});
    __syncthreads();
    // strides 16, 8, 4 over the waves, then 2, 1 over the quad: output o of a
    // tile is register o % 4 of lane o / 4 (token 4 (lane / 16) + register,
    // row lane % 16). The sums are next written behind the next tile's first
    // barriers.
    const float* f = reinterpret_cast<const float*>(sums);
    auto total = [&](int tile, int o) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float p[kEWaves];
#pragma unroll
        for (int w = 0; w < kEWaves; ++w) p[w] = f[((w * 4 + j) * TT + tile) * 256 + o];
        v[j] = ((p[0] + p[4]) + (p[2] + p[6])) + ((p[1] + p[5]) + (p[3] + p[7]));
      }
      return (v[0] + v[2]) + (v[1] + v[3]);
    };
    // gate mode: rows 0-7 of a tile are gate rows, 8-15 the same up rows
    for (int i = tid_here(); i < 256 * TT; i += kEThreads) {
      const int tile = i >> 8, o = i & 255, col = (o >> 2) & 15;
      if (kMode == kBGate && col >= 8) continue;
      const float v = total(tile, o);
      const float v2 = kMode == kBGate ? total(tile, o + 32) : 0.0f;
      const int t = t0 + 16 * tile + 4 * (o >> 6) + (o & 3), r = r0 + col;
      if (t < n && r < rows) {
        int local;
        const int s = segment_of(seg, r, &local);
        const int srows = s == 0 ? seg.rows[0] : s == 1 ? seg.rows[1] : s == 2 ? seg.rows[2] : seg.rows[3];
        const size_t out = (size_t)t * srows + local;
        segment_out(seg, s)[out] = b_epilogue<kMode>(v, v2, res, out);
      }
    }
    at += step;
    if (at >= count) return;
  }
}

// What a k_bgemm launch may have rounded differently, in the
// separate-rounding order (b256_rows): groups of four waves look at
// k_bproject's regions (bproject_rows rows, kBTokens tokens per wave), 64 at a
// time, and run those that lie in such a pair of tiles. Row group g of token
// group t is group (g + 8 t) mod `groups`'s, so that the regions of one weight
// tile, of one token and of a whole matrix all spread over the chip while the
// groups at work share a token group. With nothing to do 4.6 us, a launch's
// own; everything, 12352 rows x 2048 columns x 777 tokens, 1.71 ms (11.5 T
// multiply-adds/s, k_bproject's rate). Four 2B layers of a 777-token prompt:
// 9.1 ms, 9.8 with one inexact row tile in every matrix, 32 with nothing
// exact (one block per 256 tiles, recomputing alone: 118 and 1510).
constexpr int kFixThreads = 1024, kFixGroups = kFixThreads / 256;

template <int kMode, int TT>
__global__ __launch_bounds__(kFixThreads) void k_bgemm_fix(const uint16_t* __restrict__ x, int n, int cols, Segments seg,
                                                           const uint16_t* __restrict__ w2,
                                                           const uint16_t* __restrict__ res,
                                                           const uint32_t* __restrict__ ranges) {
  using T = BGemmTile<TT>;
  constexpr int kBlockRows = bgemm_rows<kMode>(), R = bproject_rows<kMode>();
  static_assert(kBlockRows % R == 0 && T::kTokens % kBTokens == 0, "a region lies in one tile");
  const int rows = seg.rows[0] + seg.rows[1] + seg.rows[2] + seg.rows[3];
  const int tiles_t = (n + T::kTokens - 1) / T::kTokens, tiles_r = (rows + kBlockRows - 1) / kBlockRows;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int groups = (int)gridDim.x * kFixGroups, group = (int)blockIdx.x + (int)gridDim.x * (wave >> 2);
  const int groups_r = (rows + R - 1) / R, groups_t = (n + 4 * kBTokens - 1) / (4 * kBTokens);
  const int each = (groups_r + groups - 1) / groups;  // row groups per token group, at most
  for (int base = 0; base < each * groups_t; base += 64) {
    auto place = [&](int i, int* row0, int* t0) {  // the group's region i, if there is one
      const int t = i / each, turn = (group - 8 * t) % groups;
      const int g = (turn < 0 ? turn + groups : turn) + i % each * groups;
      *row0 = g * R;
      *t0 = (t * 4 + (wave & 3)) * kBTokens;
      return t < groups_t && g < groups_r && *t0 < n;
    };
    int row0, t0;
    const bool bad = place(base + lane, &row0, &t0) &&
                     !bf_products_exact(range_of(ranges, tiles_r + t0 / T::kTokens), range_of(ranges, row0 / kBlockRows));
    for (unsigned long long todo = __ballot(bad); todo; todo &= todo - 1) {
      place(base + __ffsll(todo) - 1, &row0, &t0);
      const uint16_t* w[R];
      const uint16_t* up = nullptr;
      uint16_t* out[R];
      int local[R], srows[R];
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const int s = segment_of(seg, min(row0 + k, rows - 1), &local[k]);
        w[k] = segment_w(seg, s) + (size_t)local[k] * cols;
        if (kMode == kBGate) up = w2 + (size_t)local[k] * cols;
        out[k] = segment_out(seg, s);
        srows[k] = s == 0 ? seg.rows[0] : s == 1 ? seg.rows[1] : s == 2 ? seg.rows[2] : seg.rows[3];
      }
      b256_rows<kMode>(x, n, cols, w, up, t0, [&](int k, int t, float v, float v2) {
        if (row0 + k >= rows) return;
        const size_t o = (size_t)t * srows[k] + local[k];
        out[k][o] = b_epilogue<kMode>(v, v2, res, o);
      });
    }
  }
}

}  // namespace cq35
