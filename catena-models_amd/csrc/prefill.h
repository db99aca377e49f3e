// Batched prefill: the reference's multi-token path for key_dim 128
// (text-dispatch -> text-batch, prefill.rs:36-653). Every layer runs over all
// tokens of a chunk before the next layer. Per-token operations keep the
// decode arithmetic (they are the same reference programs with a token index):
// RMSNorm rows, convolution + L2 with history reads before the history commit,
// the DeltaNet scan over the F32 state, gated norm, head norm + RoPE + KV
// append, staged attention per query, router and top-k. The projections use
// the batched order B256: reference lane l (of 256) visits pairs l, l+256, ...
// with ONE accumulator, acc = (acc + x.lo*w.lo) + x.hi*w.hi
// (batch_projection.hex:4-18 with numeric.hex:17-28), then the 256-wide
// halving tree (cooperative.hex:285-335).
//
// Wave mapping of B256: physical lane q holds reference lanes 4q..4q+3, so
// its 16-byte quads q, q+64, q+128, ... are exactly those lanes' pairs in
// visiting order; reference strides 128..4 are physical strides 32..1
// (tree_levels<64>), strides 2 and 1 are in-lane.
#pragma once

#include "layers.h"

namespace cq35 {

constexpr int kBTokens = 8;   // tokens per wave sharing each weight quad
constexpr int kBKeyDim = 128;  // DeltaNet key width of batched calls (others run token by token)
// Tokens per chunk (buffer rows), exact and with matrix-core components: each
// chunk streams every weight once, expert weights above all (1.6 GB a 35B
// layer), and a short last chunk fills few tiles. Eight layers, whole call:
// exact 35B, 512 tokens 21.7 ms at 256 rows, 19.5 here; exact 2B, 777 tokens
// 19.5 and 17.0; matrix 35B, 4000 tokens 32.3 ms at 1024 rows, 26.8 here. A
// 35B row takes 0.16 MB.
constexpr int64_t kBChunk = 1024;
constexpr int64_t kMChunk = 2048;
// Where memory is short.
constexpr int64_t kBFewRows = 256;
constexpr int64_t kMFewRows = 1024;

__device__ __forceinline__ void b256_acc(float (&a)[4], const u32x4& x, const u32x4& w) {
  a[0] = (a[0] + lo2f(x.x) * lo2f(w.x)) + hi2f(x.x) * hi2f(w.x);
  a[1] = (a[1] + lo2f(x.y) * lo2f(w.y)) + hi2f(x.y) * hi2f(w.y);
  a[2] = (a[2] + lo2f(x.z) * lo2f(w.z)) + hi2f(x.z) * hi2f(w.z);
  a[3] = (a[3] + lo2f(x.w) * lo2f(w.w)) + hi2f(x.w) * hi2f(w.w);
}

// Tree over the 256 reference lanes; every lane of the wave must call it.
// The total is valid in lane 0.
__device__ __forceinline__ float b256_tree(const float (&a)[4]) {
  float v0 = a[0], v1 = a[1], v2 = a[2], v3 = a[3];
  tree_levels<64>(v0, v1, v2, v3);
  v0 += v2;
  v1 += v3;
  return v0 + v1;
}

// Two B256 trees at once (tree64_pair4_end: every sum with b256_tree's
// operands): a's total in lane 31, b's in lane 63.
__device__ __forceinline__ float b256_tree2(const float (&a)[4], const float (&b)[4]) {
  return tree64_pair4_end(a, b);
}

enum { kBPlain = 0, kBResidual = 1, kBGate = 2 };

// out[t][row] for `rows` outputs of `n` token rows of width `cols`
// (batch.project / batch.residual / batch.gate, batch_projection.hex:30-279,
// 280-530, 531-854). Block (bproject_rows rows, 32-token group): wave w takes
// tokens [32*by + 8w, +8) and shares each weight quad across them. Epilogues:
// bf16(total); bf16(bf16(total) (+) res); bf16(bf16(silu(bf16 g))) (x) bf16(u).
// Requires cols % 8 == 0.
// kBRows output rows per block (plain and residual modes: each wave takes
// them all, its token quads shared by the rows; gate mode: one row).
template <int kMode>
constexpr int bproject_rows() { return kMode == kBGate ? 1 : 2; }

// One wave's B256 sums of R rows (gate mode: a gate row of w and an up row of
// w2) over the tokens t0 .. t0 + kBTokens - 1 below n: emit(row k, token,
// total, up total) on lane 0.
template <int kMode, typename Emit>
__device__ __forceinline__ void b256_rows(const uint16_t* __restrict__ x, int n, int cols,
                                          const uint16_t* const (&w)[bproject_rows<kMode>()], const uint16_t* w2, int t0,
                                          Emit emit) {
  constexpr int R = bproject_rows<kMode>();
  const int lane = threadIdx.x & 63;
  const int quads = cols >> 3;
  const u32x4* wr[R];
#pragma unroll
  for (int k = 0; k < R; ++k) wr[k] = reinterpret_cast<const u32x4*>(w[k]);
  const u32x4* wr2 = reinterpret_cast<const u32x4*>(w2);
  float acc[R][kBTokens][4], acc2[kMode == kBGate ? kBTokens : 1][4];
#pragma unroll
  for (int t = 0; t < kBTokens; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int k = 0; k < R; ++k) acc[k][t][r] = 0.0f;
      if (kMode == kBGate) acc2[t][r] = 0.0f;
    }
  for (int qi = lane; qi < quads; qi += 64) {
    u32x4 wq[R];
#pragma unroll
    for (int k = 0; k < R; ++k) wq[k] = wr[k][qi];
    u32x4 wq2;
    if (kMode == kBGate) wq2 = wr2[qi];
#pragma unroll
    for (int t = 0; t < kBTokens; ++t) {
      if (t0 + t < n) {
        const u32x4 xq = reinterpret_cast<const u32x4*>(x + (size_t)(t0 + t) * cols)[qi];
#pragma unroll
        for (int k = 0; k < R; ++k) b256_acc(acc[k][t], xq, wq[k]);
        if (kMode == kBGate) b256_acc(acc2[kMode == kBGate ? t : 0], xq, wq2);
      }
    }
  }
  // totals: rows in pairs (or the gate and up sums) through b256_tree2
  float tot[R][kBTokens], tot2[kBTokens];
#pragma unroll
  for (int t = 0; t < kBTokens; ++t) {
    if (t0 + t >= n) break;  // wave-uniform
    if (kMode == kBGate) {
      const float both = b256_tree2(acc[0][t], acc2[kMode == kBGate ? t : 0]);
      tot[0][t] = lane_value(both, 31);
      tot2[t] = lane_value(both, 63);
    } else {
#pragma unroll
      for (int k = 0; k + 1 < R; k += 2) {
        const float both = b256_tree2(acc[k][t], acc[k + 1][t]);
        tot[k][t] = lane_value(both, 31);
        tot[k + 1][t] = lane_value(both, 63);
      }
      if (R % 2) tot[R - 1][t] = b256_tree(acc[R - 1][t]);
    }
  }
#pragma unroll
  for (int k = 0; k < R; ++k)
#pragma unroll
    for (int t = 0; t < kBTokens; ++t) {
      if (t0 + t >= n) break;  // wave-uniform
      if (lane == 0) emit(k, t0 + t, tot[k][t], kMode == kBGate ? tot2[t] : 0.0f);
    }
}

// The epilogues over the totals of output element o.
template <int kMode>
__device__ __forceinline__ uint16_t b_epilogue(float v, float v2, const uint16_t* res, size_t o) {
  if (kMode == kBPlain) return f2bf(v);
  if (kMode == kBResidual) return bf_add(f2bf(v), res[o]);
  return bf_mul(f2bf(silu(rbf(v))), f2bf(v2));
}

template <int kMode>
__global__ __launch_bounds__(kBlock) void k_bproject(const uint16_t* __restrict__ x, int n,
                                                     int cols, const uint16_t* __restrict__ w,
                                                     const uint16_t* __restrict__ w2, int rows,
                                                     const uint16_t* __restrict__ res,
                                                     uint16_t* __restrict__ out) {
  constexpr int R = bproject_rows<kMode>();
  const int wave = threadIdx.x >> 6;
  const int row0 = blockIdx.x * R;
  const int t0 = (blockIdx.y * 4 + wave) * kBTokens;
  if (t0 >= n || row0 >= rows) return;  // wave-uniform
  const uint16_t* wr[R];
#pragma unroll
  for (int k = 0; k < R; ++k) wr[k] = w + (size_t)min(row0 + k, rows - 1) * cols;
  b256_rows<kMode>(x, n, cols, wr, kMode == kBGate ? w2 + (size_t)row0 * cols : nullptr, t0,
                   [&](int k, int t, float total, float total2) {
                     if (row0 + k >= rows) return;
                     const size_t o = (size_t)t * rows + row0 + k;
                     out[o] = b_epilogue<kMode>(total, total2, res, o);
                   });
}

// Embedding rows of tokens [first, first + m) of the call (prefill.embed,
// qwen35_prefill.hex:69-108); block 0 clears the argmax key when asked.
__global__ __launch_bounds__(kBlock) void k_bembed(const uint64_t* __restrict__ params, int first,
                                                    const uint16_t* __restrict__ table, int hidden,
                                                    uint16_t* __restrict__ h,
                                                    unsigned long long* __restrict__ best) {
  const uint64_t token = params[1 + first + blockIdx.x];
  const uint16_t* row = table + token * (uint64_t)hidden;
  uint16_t* dst = h + (size_t)blockIdx.x * hidden;
  for (int i = threadIdx.x; i < hidden; i += blockDim.x) dst[i] = row[i];
  if (blockIdx.x == 0 && threadIdx.x == 0 && best) *best = 0ull;
}

// RMSNorm of each row (qwen35.normalize with rows = sequence,
// qwen35.hex:912-977): one block per row, the decode norm's arithmetic.
__global__ __launch_bounds__(kBlock) void k_bnorm(const uint16_t* __restrict__ x,
                                                   const float* __restrict__ w, int cols, float eps,
                                                   uint16_t* __restrict__ out) {
  extern __shared__ __align__(16) u32x4 bn_xs[];
  __shared__ float red[4];
  const uint16_t* xr = x + (size_t)blockIdx.x * cols;
  NormIn nin;
  norm_prefetch(nin, xr, w, cols);
  norm_finish(nin, bn_xs, xr, w, cols, eps, red);
  u32x4* o = reinterpret_cast<u32x4*>(out + (size_t)blockIdx.x * cols);
  for (int i = threadIdx.x; i < (cols >> 3); i += blockDim.x) o[i] = bn_xs[i];
}

// Four-tap convolution of every token of the chunk, then the per-head L2
// norm of the Q and K heads (batch.prepare, batch_prepare.hex:3-158): the tap
// at position p < `first` reads the cache history slot p % 3 (still holding
// the rows before this chunk), later taps read the chunk's own rows.
//
// Block (KD channels, TB tokens), a thread two channels of TB / 4 consecutive
// tokens: each row is read once per thread (and three rows before its first),
// the serial sum of squares of a token's head runs on a lane of its own, all
// tokens at once (one block per token left 255 threads waiting for it: 1024
// tokens of a 35B layer 70 us, now 30). TB 8 for short calls, where a thread's
// tokens in turn would be the time (37 tokens: 6 us, 10 at TB 32).
constexpr int kPrepareTokens = 32, kPrepareFew = 8;

template <int TB>
__global__ __launch_bounds__(kBlock) void k_bprepare(
    const uint16_t* __restrict__ qkv, const uint16_t* __restrict__ cache, int64_t conv_base,
    const uint64_t* __restrict__ params, int first, int m, const float* __restrict__ conv_w, int qkv_size,
    int key_heads, uint16_t* __restrict__ conv_out, uint16_t* __restrict__ q_out,
    uint16_t* __restrict__ k_out) {
  constexpr int KD = kBKeyDim, kPairs = KD / 2, kGroups = kBlock / kPairs, kEach = TB / kGroups;
  static_assert(kBlock % kPairs == 0 && TB % kGroups == 0, "channel pairs");
  __shared__ float squares[TB][KD + 1];
  __shared__ float total[TB];
  const int64_t begin = (int64_t)params[0] + first;  // position of the chunk's row 0
  const int chunk = blockIdx.x, pair = threadIdx.x % kPairs, group = threadIdx.x / kPairs;
  const int t0 = blockIdx.y * TB + group * kEach;
  const int ch = chunk * KD + 2 * pair;
  const bool active = ch < qkv_size;
  const int key_size = key_heads * KD;
  const bool heads = chunk < 2 * key_heads;  // value heads: convolution only
  auto row = [&](int t) -> uint32_t {        // the chunk's row t, or the history before it
    const int64_t p = begin + t;
    if (p < 0) return 0u;
    const uint16_t* r = t < 0 ? cache + conv_base + (p % 3) * qkv_size : qkv + (size_t)t * qkv_size;
    return *reinterpret_cast<const uint32_t*>(r + ch);
  };
  float value[kEach][2];
  if (active && t0 < m) {
    const f32x4 w0 = reinterpret_cast<const f32x4*>(conv_w)[ch], w1 = reinterpret_cast<const f32x4*>(conv_w)[ch + 1];
    uint32_t in[kEach + 3];
#pragma unroll
    for (int i = 0; i < kEach + 3; ++i) in[i] = row(min(t0 - 3 + i, m - 1));
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      auto conv = [&](auto half, const f32x4& w) {
        auto x = [&](int k) { return decltype(half)::value ? hi2f(in[i + k]) : lo2f(in[i + k]); };
        const float sum = (x(0) * w[0] + x(2) * w[2]) + (x(1) * w[1] + x(3) * w[3]);
        return f2bf(silu(rbf(sum)));
      };
      const uint16_t lo = conv(std::false_type{}, w0), hi = conv(std::true_type{}, w1);
      if (t0 + i < m) *reinterpret_cast<uint32_t*>(conv_out + (size_t)(t0 + i) * qkv_size + ch) = pack_bf(lo, hi);
      value[i][0] = bf2f(lo);
      value[i][1] = bf2f(hi);
      if (heads) {
        squares[group * kEach + i][2 * pair] = value[i][0] * value[i][0];
        squares[group * kEach + i][2 * pair + 1] = value[i][1] * value[i][1];
      }
    }
  }
  if (!heads) return;  // uniform
  __syncthreads();
  if (threadIdx.x < TB && blockIdx.y * TB + (int)threadIdx.x < m) {
    float s = 0.0f;
#pragma unroll 16
    for (int i = 0; i < KD; ++i) s += squares[threadIdx.x][i];
    total[threadIdx.x] = nsqrt(s + bitsf(0x358637bdu));
  }
  __syncthreads();
  uint16_t* dst = (chunk < key_heads ? q_out : k_out) + (chunk % key_heads) * KD + 2 * pair;
#pragma unroll
  for (int i = 0; i < kEach; ++i) {
    if (t0 + i >= m) break;
    const float norm = total[group * kEach + i];
    *reinterpret_cast<uint32_t*>(dst + (size_t)(t0 + i) * key_size) =
        pack_bf(f2bf(value[i][0] / norm), f2bf(value[i][1] / norm));
  }
}

// k_gated_norm (layers.h) over the chunk's (token, head) rows of value_dim
// contiguous values: `per` (at most kGatedRows) rows per block, a row's serial
// sum of squares on a lane of its own, the rest eight values at a time. One
// block per row left 255 threads waiting for that sum: 1024 tokens of a 35B
// layer 34 us, now 16. value_dim % 8 == 0, at most 256.
constexpr int kGatedRows = 32;
inline size_t bgated_lds_bytes(int value_dim) { return (size_t)kGatedRows * (value_dim + 2) * 4; }

__global__ __launch_bounds__(kBlock) void k_bgated_norm(const uint16_t* __restrict__ core,
                                                        const uint16_t* __restrict__ z, const float* __restrict__ w,
                                                        int rows, int per, int value_dim, float eps,
                                                        uint16_t* __restrict__ out) {
  extern __shared__ float bgn_lds[];
  float* squares = bgn_lds;  // [row][value_dim + 1]
  float* rms = bgn_lds + kGatedRows * (value_dim + 1);
  const int r0 = blockIdx.x * per, quads = value_dim >> 3;
  const int count = min(per, rows - r0) * quads;
  const size_t base = (size_t)r0 * quads;
  for (int i = threadIdx.x; i < count; i += kBlock) {
    const u32x4 v = ldq(core, base + i);
    float* s = squares + (i / quads) * (value_dim + 1) + 8 * (i % quads);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[2 * e] = lo2f(v[e]) * lo2f(v[e]);
      s[2 * e + 1] = hi2f(v[e]) * hi2f(v[e]);
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < min(per, rows - r0)) {
    float s = 0.0f;
#pragma unroll 8
    for (int i = 0; i < value_dim; ++i) s += squares[threadIdx.x * (value_dim + 1) + i];
    rms[threadIdx.x] = nsqrt(s / (float)value_dim + eps);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < count; i += kBlock) {
    const u32x4 v = ldq(core, base + i), zq = ldq(z, base + i);
    const float d = rms[i / quads];
    const f32x4* wq = reinterpret_cast<const f32x4*>(w) + 2 * (i % quads);
    const f32x4 wl = wq[0], wh = wq[1];
    u32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = e < 2 ? wl[2 * e] : wh[2 * e - 4], b = e < 2 ? wl[2 * e + 1] : wh[2 * e - 3];
      y[e] = pack_bf(f2bf((lo2f(v[e]) / d * a) * silu(lo2f(zq[e]))), f2bf((hi2f(v[e]) / d * b) * silu(hi2f(zq[e]))));
    }
    reinterpret_cast<u32x4*>(out)[base + i] = y;
  }
}

// History commit after the chunk's reads: the last min(m, 3) raw QKV rows
// into slots position % 3 (batch.history, batch_prepare.hex:209-292).
__global__ __launch_bounds__(kBlock) void k_bhistory(const uint16_t* __restrict__ qkv, int m,
                                                      uint16_t* __restrict__ cache,
                                                      int64_t conv_base,
                                                      const uint64_t* __restrict__ params,
                                                      int first, int qkv_size) {
  const int kept = m < 3 ? m : 3;
  const int64_t begin = (int64_t)params[0] + first;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < (int64_t)kept * qkv_size;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int t = m - kept + (int)(i / qkv_size);
    const int ch = (int)(i % qkv_size);
    cache[conv_base + ((begin + t) % 3) * qkv_size + ch] = qkv[(size_t)t * qkv_size + ch];
  }
}

// Sum over the 32 lanes of each half wave, the total in every lane: the
// halving tree's operands (strides 16 ... 1; a lane past the first s of a
// level adds the same two values the other way round).
__device__ __forceinline__ float sum32_everywhere(float v) {
  const int b = __builtin_bit_cast(int, v);
  const auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);  // a half's first row, its second
  v = __builtin_bit_cast(float, (int)r[0]) + __builtin_bit_cast(float, (int)r[1]);
  auto turned = [](float x, auto ror) {
    const int i = __builtin_bit_cast(int, x);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, 0x120 + decltype(ror)::value, 0xf, 0xf, true));
  };
  v += turned(v, std::integral_constant<int, 8>{});
  v += turned(v, std::integral_constant<int, 4>{});
  v += turned(v, std::integral_constant<int, 2>{});
  v += turned(v, std::integral_constant<int, 1>{});
  return v;
}

// DeltaNet scan over the chunk's tokens with the F32 state in registers
// (batch.scan, batch_scan.hex:1-200): per token exactly the single-step
// arithmetic of k_delta (32 lanes per value channel, lane l owns key elements
// l, l+32, ...; serial from 0.0, 32-wide halving tree), 8 channels of one head
// per block. Requires value_dim % 8 == 0.
//
// Bound: instruction issue of a token's serial chain (two sums over 32
// reference lanes, the state update between them). The chain holds nothing
// else: per stage of kScanTokens tokens the block first stages the head's k
// and q rows widened to F32, its channels' values, and every token's decay
// and rate (the next stage's rows are requested before the chain starts); a
// token's values are read from LDS a token ahead; the sums leave their total
// in every lane; lane t keeps token t's output, and scale, rounding and store
// run once per stage: 67 vector instructions a token. 2048 tokens of a 35B
// layer take 443 us; 1024 of them 225 before the gates went first (355 with
// BF16 rows widened and the totals broadcast inside the chain; 16 lanes per
// channel, a quarter fewer instructions but one wave per SIMD: 218).
constexpr int kScanTokens = 32;

constexpr size_t kScanLds = (size_t)kScanTokens * kBKeyDim * 2 * 4 + (size_t)kScanTokens * 8 + (size_t)kScanTokens * 8 * (4 + 2);

__global__ __launch_bounds__(kBlock) void k_bscan(
    const uint16_t* __restrict__ conv, const uint16_t* __restrict__ q,
    const uint16_t* __restrict__ k, const uint16_t* __restrict__ alpha,
    const uint16_t* __restrict__ beta, const float* __restrict__ dt, const float* __restrict__ a,
    float* __restrict__ state, int m, int value_size, int value_dim, int value_heads, int key_heads, int qkv_size,
    float scale, uint16_t* __restrict__ out) {
  constexpr int key_dim = kBKeyDim, KJ = key_dim / 32, quads = key_dim / 8;  // KJ key elements per lane
  constexpr int CH = kBlock / 32;  // channels
  constexpr int kRows = kScanTokens * quads / kBlock;  // quads of k and of q per thread and stage
  static_assert(kScanTokens == 32 && kScanTokens * CH == kBlock && kRows * kBlock == kScanTokens * quads, "a token per lane, a value per thread");
  extern __shared__ __align__(16) unsigned char scan_lds[];
  float* sk = reinterpret_cast<float*>(scan_lds);
  float* sq = sk + kScanTokens * key_dim;
  float2* sgate = reinterpret_cast<float2*>(sq + kScanTokens * key_dim);  // decay, rate
  float* sval = reinterpret_cast<float*>(sgate + kScanTokens);            // [token][CH]
  uint16_t* sout = reinterpret_cast<uint16_t*>(sval + kScanTokens * CH);  // [token][CH]
  const int c0 = blockIdx.x * CH;
  const int ch = threadIdx.x / 32;
  const int c = c0 + ch;
  const int lane = threadIdx.x % 32;
  const int head = c0 / value_dim;
  const int kbase = (head % key_heads) * key_dim;
  const int key_size = key_heads * key_dim;
  const float dth = dt[head], ah = a[head];
  float s[KJ];
#pragma unroll
  for (int j = 0; j < KJ; ++j) s[j] = state[(size_t)c * key_dim + lane + 32 * j];
  u32x4 kq4[kRows], qq4[kRows];
  uint16_t val, al, be;
  // a stage's rows into registers (rows past the last repeat it)
  auto request = [&](int t0) {
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const int idx = threadIdx.x + kBlock * r;
      const int t = min(t0 + idx / quads, m - 1);
      const size_t src = (size_t)t * key_size + kbase + 8 * (idx % quads);
      kq4[r] = *reinterpret_cast<const u32x4*>(k + src);
      qq4[r] = *reinterpret_cast<const u32x4*>(q + src);
    }
    val = conv[(size_t)min(t0 + (int)threadIdx.x / CH, m - 1) * qkv_size + 2 * key_size + c0 + threadIdx.x % CH];
    const int t = min(t0 + lane, m - 1);
    al = alpha[(size_t)t * value_heads + head];
    be = beta[(size_t)t * value_heads + head];
  };
  // the gates' chain of the first wave ahead of the rows that all widen (443
  // against 456 us per 2048 tokens of a 35B layer the other way round)
  auto place = [&]() {
    sval[threadIdx.x] = bf2f(val);
    if (threadIdx.x < kScanTokens) {
      const float time_step = softplus(bf2f(al) + dth);
      sgate[threadIdx.x] = float2{hexp(rbf(time_step * ah)), rbf(sigmoid(bf2f(be)))};
    }
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const int idx = threadIdx.x + kBlock * r;
      auto widen = [&](float* to, const u32x4& v) {
        f32x4* d = reinterpret_cast<f32x4*>(to + 8 * idx);
        d[0] = f32x4{lo2f(v.x), hi2f(v.x), lo2f(v.y), hi2f(v.y)};
        d[1] = f32x4{lo2f(v.z), hi2f(v.z), lo2f(v.w), hi2f(v.w)};
      };
      widen(sk, kq4[r]);
      widen(sq, qq4[r]);
    }
  };
  struct Token {
    float k[KJ], q[KJ], value;
    float2 gate;
  };
  auto read = [&](int tt, Token& v) {
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      v.k[j] = sk[tt * key_dim + lane + 32 * j];
      v.q[j] = sq[tt * key_dim + lane + 32 * j];
    }
    v.value = sval[tt * CH + ch];
    v.gate = sgate[tt];
  };
  float kept = 0.0f;
  auto chain = [&](int tt, const Token& v) {
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < KJ; ++j) acc += s[j] * v.k[j];
    const float total = sum32_everywhere(acc);
    const float delta = (v.value - total * v.gate.x) * v.gate.y;
    float acc2 = 0.0f;
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      s[j] = s[j] * v.gate.x + v.k[j] * delta;
      acc2 += s[j] * v.q[j];
    }
    acc2 = sum32_everywhere(acc2);
    kept = tt == lane ? acc2 : kept;
  };
  request(0);
  for (int t0 = 0; t0 < m; t0 += kScanTokens) {
    const int ts = min(kScanTokens, m - t0);
    place();
    if (t0 + kScanTokens < m) request(t0 + kScanTokens);
    __syncthreads();
    Token x, y;
    read(0, x);
    int tt = 0;
#pragma unroll 1
    for (; tt + 2 <= ts; tt += 2) {
      read(tt + 1, y);
      chain(tt, x);
      read(min(tt + 2, kScanTokens - 1), x);
      chain(tt + 1, y);
    }
    if (tt < ts) chain(tt, x);
    sout[lane * CH + ch] = f2bf(kept * scale);
    __syncthreads();
    if ((int)threadIdx.x < ts)
      *reinterpret_cast<u32x4*>(out + (size_t)(t0 + threadIdx.x) * value_size + c0) =
          reinterpret_cast<const u32x4*>(sout)[threadIdx.x];
  }
#pragma unroll
  for (int j = 0; j < KJ; ++j) state[(size_t)c * key_dim + lane + 32 * j] = s[j];
}

// RoPE tables [cos x R/2 | sin x R/2] for the chunk's positions
// (qwen3.rope-frequency + rope-sincos, batch_full_prepare.hex:63-70).
__global__ __launch_bounds__(kBlock) void k_brope(const uint64_t* __restrict__ params, int first,
                                                   const float* __restrict__ freq, int half,
                                                   float* __restrict__ rope) {
  const float position = (float)(uint32_t)((int64_t)params[0] + first + blockIdx.x);
  float* r = rope + (size_t)blockIdx.x * 2 * half;
  for (int i = threadIdx.x; i < half; i += blockDim.x) {
    float s, c;
    sincos_q(position * freq[i], &s, &c);
    r[i] = c;
    r[half + i] = s;
  }
}

// MoE router logits of every token (batch.moe.router, batch_moe.hex:45-135):
// the decode router's S32 over the normalised row with F32 weights, rows
// [0, E) routed and row E the shared-expert gate. Block (4 rows, token).
__global__ __launch_bounds__(kBlock) void k_brouter(const uint16_t* __restrict__ x, int cols,
                                                     const float* __restrict__ w,
                                                     const float* __restrict__ shared_w,
                                                     int experts, float* __restrict__ logits) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int rows = experts + 1;
  const int row = blockIdx.x * 4 + wave;
  const int t = blockIdx.y;
  const int rc = min(row, rows - 1);
  const float* wr = rc < experts ? w + (size_t)rc * cols : shared_w;
  const uint16_t* xr = x + (size_t)t * cols;
  // physical lane l = 2r + h: reference lane r's low (h = 0) or high (h = 1)
  // accumulator over elements l + 64k
  float acc = 0.0f;
  for (int i = lane; i < cols; i += 64) acc += bf2f(xr[i]) * wr[i];
  float v = acc + lane_down<1>(acc);
  v += lane_down<32>(v);
  v += lane_down<16>(v);
  v += lane_down<8>(v);
  v += lane_down<4>(v);
  v += lane_down<2>(v);
  if (lane == 0 && row < rows) logits[(size_t)t * rows + row] = v;
}

// k_brouter's logits with each weight row read once per 16 tokens: wave w of
// block (row group, token group) keeps rows 16 rg + 2 w and + 1 in registers
// (lane l: elements l + 64 k), the group's 16 token rows are staged in LDS,
// and every (row, token) sum runs in k_brouter's order (each lane's chain
// over k, then the same tree), so the logits are bit-identical. cols a
// multiple of 64, at most 2048.
constexpr int kRouterTokens = 16;
constexpr int kRouterRows = 16;  // 2 per wave, 8 waves
template <int KJ>  // cols / 64
__global__ __launch_bounds__(512) void k_brouter_shared(const uint16_t* __restrict__ x, int n,
                                                        const float* __restrict__ w,
                                                        const float* __restrict__ shared_w, int experts,
                                                        float* __restrict__ logits) {
  constexpr int cols = 64 * KJ;
  __shared__ uint16_t xs[kRouterTokens][cols];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int rows = experts + 1;
  const int t0 = blockIdx.y * kRouterTokens;
  const int tn = min(kRouterTokens, n - t0);
  float wv[2][KJ];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int rc = min(blockIdx.x * kRouterRows + 2 * wave + r, rows - 1);
    const float* wr = rc < experts ? w + (size_t)rc * cols : shared_w;
#pragma unroll
    for (int k = 0; k < KJ; ++k) wv[r][k] = wr[lane + 64 * k];
  }
  constexpr int pieces = cols / 8;
  for (int i = threadIdx.x; i < tn * pieces; i += blockDim.x) {
    const int t = i / pieces, p = i - t * pieces;
    reinterpret_cast<u32x4*>(&xs[t][0])[p] = ldq(x + (size_t)(t0 + t) * cols, p);
  }
  __syncthreads();
  for (int t = 0; t < tn; ++t) {
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      float acc = 0.0f;
#pragma unroll
      for (int k = 0; k < KJ; ++k)
        acc += bf2f(xs[t][lane + 64 * k]) * wv[r][k];
      float v = acc + lane_down<1>(acc);
      v += lane_down<32>(v);
      v += lane_down<16>(v);
      v += lane_down<8>(v);
      v += lane_down<4>(v);
      v += lane_down<2>(v);
      const int row = blockIdx.x * kRouterRows + 2 * wave + r;
      if (lane == 0 && row < rows) logits[(size_t)(t0 + t) * rows + row] = v;
    }
  }
}

// Top-k of each token's routed logits by the reference's rank,
// rank(e) = #{i : l_i > l_e} + #{i < e : !(l_e > l_i)}, and the softmax
// weights p_j = exp(l_j - l_0) / den with den summed left to right
// (batch.moe.select, batch_moe.hex:136-317). One block per token. With
// last_ids, the last token's ids are also written there (the layer's slot of
// the session's exported top-k).
__global__ __launch_bounds__(kBlock) void k_bselect(const float* __restrict__ logits, int experts,
                                                     int top_k, int* __restrict__ ids,
                                                     float* __restrict__ probs, int* __restrict__ last_ids) {
  extern __shared__ float bs_lg[];
  __shared__ float chosen[64];
  const int t = blockIdx.x;
  const float* lt = logits + (size_t)t * (experts + 1);
  for (int e = threadIdx.x; e < experts; e += blockDim.x) bs_lg[e] = lt[e];
  // NaN logits can make ranks collide: the largest expert index of a shared
  // rank takes it (the restatement's ascending scatter; an LDS maximum) and
  // an unassigned rank k keeps expert k; without NaNs the ranks are a
  // permutation.
  __shared__ int won[64];
  if (threadIdx.x < top_k) won[threadIdx.x] = -1;
  __syncthreads();
  for (int e = threadIdx.x; e < experts; e += blockDim.x) {
    const float le = bs_lg[e];
    int rank = 0;
    for (int i = 0; i < experts; ++i) {
      const float o = bs_lg[i];
      rank += (o > le) ? 1 : ((i < e && !(le > o)) ? 1 : 0);
    }
    if (rank < top_k) atomicMax(&won[rank], e);
  }
  __syncthreads();
  if (threadIdx.x < top_k) {
    const int e = won[threadIdx.x] >= 0 ? won[threadIdx.x] : threadIdx.x;
    ids[(size_t)t * top_k + threadIdx.x] = e;
    chosen[threadIdx.x] = bs_lg[e];
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    const float ex = lane < top_k ? hexp(chosen[lane] - chosen[0]) : 0.0f;
    float den = 0.0f;
    for (int j = 0; j < top_k; ++j) den = den + __shfl(ex, j, 64);
    if (lane < top_k) probs[(size_t)t * top_k + lane] = ex / den;
  }
  if (last_ids && t == (int)gridDim.x - 1 && threadIdx.x < top_k)
    last_ids[threadIdx.x] = ids[(size_t)t * top_k + threadIdx.x];
}

// Expert gate/up of every token (batch.moe.gate, batch_moe.hex:339-411):
// dual B256 over the normalised row; routed rows r < K*I use expert
// ids[slot = r / I], row r % I, and give bf16(silu(g)*u*p_slot); shared rows
// give bf16(bf16(bf16(silu(g))*u)*sigmoid(l_E)), with g, u the bf16 totals.
// Block (4 rows, token). Requires hidden % 8 == 0.
__global__ __launch_bounds__(kBlock) void k_bmoe_gate(
    const uint16_t* __restrict__ x, int hidden, const uint16_t* __restrict__ gate,
    const uint16_t* __restrict__ up, const uint16_t* __restrict__ sgate,
    const uint16_t* __restrict__ sup, const int* __restrict__ ids, const float* __restrict__ probs,
    const float* __restrict__ logits, int experts, int top_k, int inter, int shared_inter,
    uint16_t* __restrict__ active) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = blockIdx.y;
  const int rows = top_k * inter + shared_inter;
  const int r = blockIdx.x * 4 + wave;
  if (r >= rows) return;  // wave-uniform
  const bool routed = r < top_k * inter;
  const int slot = routed ? r / inter : 0;
  const uint16_t *wg, *wu;
  if (routed) {
    const size_t wrow = (size_t)ids[(size_t)t * top_k + slot] * inter + r % inter;
    wg = gate + wrow * hidden;
    wu = up + wrow * hidden;
  } else {
    wg = sgate + (size_t)(r - top_k * inter) * hidden;
    wu = sup + (size_t)(r - top_k * inter) * hidden;
  }
  const u32x4* xq = reinterpret_cast<const u32x4*>(x + (size_t)t * hidden);
  const u32x4* gq = reinterpret_cast<const u32x4*>(wg);
  const u32x4* uq = reinterpret_cast<const u32x4*>(wu);
  float ag[4] = {0.0f, 0.0f, 0.0f, 0.0f}, au[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int qi = lane; qi < (hidden >> 3); qi += 64) {
    const u32x4 xv = xq[qi];
    b256_acc(ag, xv, gq[qi]);
    b256_acc(au, xv, uq[qi]);
  }
  const float both = b256_tree2(ag, au);
  const float g = lane_value(both, 31), u = lane_value(both, 63);
  if (lane == 0) {
    const float gb = rbf(g), ub = rbf(u);
    const float activated = silu(gb);
    float y;
    if (routed) {
      y = (activated * ub) * probs[(size_t)t * top_k + slot];
    } else {
      const float shared_prob = sigmoid(logits[(size_t)t * (experts + 1) + experts]);
      y = rbf(rbf(activated) * ub) * shared_prob;
    }
    active[(size_t)t * rows + r] = f2bf(y);
  }
}

// k_bmoe_gate with the weights read once per chunk: the (token, slot)
// assignments bucketed by expert (k_moe_bucket), block = kGRows rows of
// expert blockIdx.y, each wave kGRowsPerWave of them with their gate and up
// quads (lane + 64 j) held in registers, applied to the expert's tokens in
// turn (the next token's input quads in flight); the epilogues of up to 64
// tokens run at once, one per lane. kShared: the shared expert
// over tokens [16 blockIdx.y, +16). Per (token, row) the arithmetic is
// k_bmoe_gate's: the B256 lane order over the quads, the tree and the
// epilogue, so the results are the same bits.
constexpr int kGRowsPerWave = 1;
constexpr int kGRows = 4 * kGRowsPerWave;  // rows per block
constexpr int kGSharedTokens = 16;

template <int NQ, bool kShared>
__global__ __launch_bounds__(kBlock) void k_bmoe_gate_grouped(
    const uint16_t* __restrict__ x, int hidden, const uint16_t* __restrict__ gate,
    const uint16_t* __restrict__ up, const int* __restrict__ eoff, const int* __restrict__ order,
    const float* __restrict__ probs, const float* __restrict__ logits, int experts, int top_k, int inter,
    int shared_inter, int n, uint16_t* __restrict__ active) {
  constexpr int RW = kGRowsPerWave;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int width = kShared ? shared_inter : inter;
  const int r0 = blockIdx.x * kGRows + RW * wave;
  if (r0 >= width) return;  // wave-uniform
  const int e = kShared ? 0 : blockIdx.y;
  const int begin = kShared ? kGSharedTokens * blockIdx.y : eoff[e];
  const int count = kShared ? min(kGSharedTokens, n - begin) : eoff[e + 1] - begin;
  if (count <= 0) return;
  const int quads = hidden >> 3;
  const int rows = top_k * inter + shared_inter;
  u32x4 gw[RW][NQ], uw[RW][NQ];
#pragma unroll
  for (int k = 0; k < RW; ++k) {
    const int r = min(r0 + k, width - 1);
    const size_t wrow = kShared ? (size_t)r : (size_t)e * inter + r;
    const u32x4* gq = reinterpret_cast<const u32x4*>(gate + wrow * hidden);
    const u32x4* uq = reinterpret_cast<const u32x4*>(up + wrow * hidden);
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
      gw[k][j] = gq[min(lane + 64 * j, quads - 1)];
      uw[k][j] = uq[min(lane + 64 * j, quads - 1)];
    }
  }
  auto token = [&](int i) { return kShared ? begin + i : order[begin + i] / top_k; };
  auto load = [&](u32x4 (&xv)[NQ], int i) {
    const u32x4* xq = reinterpret_cast<const u32x4*>(x + (size_t)token(min(i, count - 1)) * hidden);
#pragma unroll
    for (int j = 0; j < NQ; ++j) xv[j] = xq[min(lane + 64 * j, quads - 1)];
  };
  // the epilogues of up to 64 tokens at once: lane j keeps the totals of
  // token (i & ~63) + j and applies k_bmoe_gate's epilogue to it
  float pg[RW], pu[RW];
  auto finish = [&](int b, int m) {
    if (lane >= m) return;
    const int i = b + lane;
    const int a = kShared ? 0 : order[begin + i];
    const int t = kShared ? begin + i : a / top_k;
#pragma unroll
    for (int k = 0; k < RW; ++k) {
      const int r = r0 + k;
      if (r >= width) continue;
      const float gb = rbf(pg[k]), ub = rbf(pu[k]);
      const float activated = silu(gb);
      if (kShared) {
        const float shared_prob = sigmoid(logits[(size_t)t * (experts + 1) + experts]);
        active[(size_t)t * rows + top_k * inter + r] = f2bf(rbf(rbf(activated) * ub) * shared_prob);
      } else {
        const int slot = a - t * top_k;
        active[(size_t)t * rows + slot * inter + r] = f2bf((activated * ub) * probs[a]);
      }
    }
  };
  auto compute = [&](const u32x4 (&xv)[NQ], int i) {
#pragma unroll
    for (int k = 0; k < RW; ++k) {
      float ag[4] = {0.0f, 0.0f, 0.0f, 0.0f}, au[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < NQ; ++j)
        if (lane + 64 * j < quads) {
          b256_acc(ag, xv[j], gw[k][j]);
          b256_acc(au, xv[j], uw[k][j]);
        }
      const float both = b256_tree2(ag, au);
      const float g = lane_value(both, 31), u = lane_value(both, 63);
      if (lane == (i & 63)) {
        pg[k] = g;
        pu[k] = u;
      }
    }
    if ((i & 63) == 63 || i == count - 1) finish(i & ~63, (i & 63) + 1);  // wave-uniform
  };
  u32x4 xa[NQ], xb[NQ];
  load(xa, 0);
#pragma unroll 1
  for (int i = 0; i < count; i += 2) {
    load(xb, i + 1);
    compute(xa, i);
    if (i + 1 < count) {
      load(xa, i + 2);
      compute(xb, i + 1);
    }
  }
}

// Expert down of every token (batch.moe.down, batch_moe.hex:453-563): B256
// over the K*I/2 routed pairs (pair p from expert ids[p / (I/2)], channel
// p % (I/2)) with the shared pairs p < SI/2 accumulated in the same lanes,
// then bf16(bf16(routed + residual) (+) bf16(shared)). Block (4 rows,
// token), numbered so that the blocks of one 4-row group, all tokens, run on
// one XCD in sequence (block b runs on XCD b mod 8; XCD x takes the groups
// x, x + 8, ... in ascending order): the group's rows of every expert, 4 KB
// each, are read from HBM once into that XCD's L2 and shared by the tokens
// routed there, instead of each token streaming its experts' whole
// matrices. Grid: 8 * n * ceil(ceil(hidden / 4) / 8) blocks. Requires
// inter % 8 == 0, shared_inter % 8 == 0 and shared_inter <= top_k * inter.
inline int bmoe_down_grid(int hidden, int n) { return 8 * n * (((hidden + 3) / 4 + 7) / 8); }

__global__ __launch_bounds__(kBlock) void k_bmoe_down(
    const uint16_t* __restrict__ active, const uint16_t* __restrict__ down,
    const uint16_t* __restrict__ sdown, const int* __restrict__ ids,
    const uint16_t* __restrict__ res, int hidden, int top_k, int inter, int shared_inter, int n,
    uint16_t* __restrict__ out) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int local = (int)(blockIdx.x >> 3);
  const int group = (int)(blockIdx.x & 7) + 8 * (local / n), t = local % n;
  const int o = group * 4 + wave;
  if (o >= hidden) return;  // wave-uniform
  const int rows = top_k * inter + shared_inter;
  const int aq = top_k * inter / 8, iq = inter / 8, sq = shared_inter / 8;
  const u32x4* xa = reinterpret_cast<const u32x4*>(active + (size_t)t * rows);
  const int* idt = ids + (size_t)t * top_k;
  const u32x4* sw = reinterpret_cast<const u32x4*>(sdown + (size_t)o * shared_inter);
  float ar[4] = {0.0f, 0.0f, 0.0f, 0.0f}, as[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int qi = lane; qi < aq; qi += 64) {
    const int slot = qi / iq, ch = qi % iq;
    const u32x4* wr =
        reinterpret_cast<const u32x4*>(down + ((size_t)idt[slot] * hidden + o) * inter);
    b256_acc(ar, xa[qi], wr[ch]);
    if (qi < sq) b256_acc(as, xa[aq + qi], sw[qi]);
  }
  const float both = b256_tree2(ar, as);
  const float routed = lane_value(both, 31), shared = lane_value(both, 63);
  if (lane == 0) {
    const size_t i = (size_t)t * hidden + o;
    out[i] = bf_add(f2bf(routed + bf2f(res[i])), f2bf(shared));
  }
}

// k_bmoe_down with each wave on kDRows consecutive output rows of one token:
// the token's activation quads are read once into registers and used for
// every row, each row's weight quads are read once. Block = (kDRows-row
// group, kDTokens tokens), wave w on token 4 by + w; blocks numbered as in
// k_bmoe_down, a group's blocks (all tokens) on one XCD in sequence. Per
// (token, row) the products, the lane chains over qi = lane, lane + 64, ...
// (routed and shared), the tree and the epilogue are k_bmoe_down's, so the
// results are the same bits. NQ: quads per lane, ceil(top_k * inter / 512)
// rounded up to a power of two.
constexpr int kDRows = 8;
constexpr int kDTokens = kBlock / 64;
inline int bmoe_down_rows_grid(int hidden, int n) {
  const int groups = (hidden + kDRows - 1) / kDRows, tiles = (n + kDTokens - 1) / kDTokens;
  return 8 * tiles * ((groups + 7) / 8);
}

template <int NQ>
__global__ __launch_bounds__(kBlock) void k_bmoe_down_rows(
    const uint16_t* __restrict__ active, const uint16_t* __restrict__ down,
    const uint16_t* __restrict__ sdown, const int* __restrict__ ids,
    const uint16_t* __restrict__ res, int hidden, int top_k, int inter, int shared_inter, int n,
    uint16_t* __restrict__ out) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles = (n + kDTokens - 1) / kDTokens;
  const int local = (int)(blockIdx.x >> 3);
  const int group = (int)(blockIdx.x & 7) + 8 * (local / tiles);
  const int t = (local % tiles) * kDTokens + wave;
  const int o0 = group * kDRows;
  if (o0 >= hidden || t >= n) return;  // wave-uniform
  const int rows = top_k * inter + shared_inter;
  const int aq = top_k * inter / 8, iq = inter / 8, sq = shared_inter / 8;
  const u32x4* xa = reinterpret_cast<const u32x4*>(active + (size_t)t * rows);
  const int* idt = ids + (size_t)t * top_k;
  u32x4 xv[NQ], xs[NQ];
  size_t woff[NQ];
#pragma unroll
  for (int j = 0; j < NQ; ++j) {
    const int qi = min(lane + 64 * j, aq - 1), slot = qi / iq, ch = qi - slot * iq;
    xv[j] = xa[qi];
    woff[j] = (size_t)idt[slot] * hidden * inter + (size_t)ch * 8;
    if (64 * j < sq) xs[j] = xa[aq + min(lane + 64 * j, sq - 1)];
  }
#pragma unroll
  for (int r = 0; r < kDRows; ++r) {
    const int o = o0 + r;
    if (o >= hidden) break;  // wave-uniform
    u32x4 wv[NQ], ws[NQ];
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
      wv[j] = *reinterpret_cast<const u32x4*>(down + woff[j] + (size_t)o * inter);
      if (64 * j < sq)
        ws[j] = reinterpret_cast<const u32x4*>(sdown + (size_t)o * shared_inter)[min(lane + 64 * j, sq - 1)];
    }
    float ar[4] = {0.0f, 0.0f, 0.0f, 0.0f}, as[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
      if (lane + 64 * j < aq) b256_acc(ar, xv[j], wv[j]);
      if (lane + 64 * j < sq) b256_acc(as, xs[j], ws[j]);
    }
    const float both = b256_tree2(ar, as);
    const float routed = lane_value(both, 31), shared = lane_value(both, 63);
    if (lane == 0) {
      const size_t i = (size_t)t * hidden + o;
      out[i] = bf_add(f2bf(routed + bf2f(res[i])), f2bf(shared));
    }
  }
}

}  // namespace cq35
