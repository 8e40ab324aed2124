// Decoder glue around the MoE call (gfx950): the hyper-connection that makes
// the MoE branch's input from the residual streams.  The injection of the
// branch output back into the streams runs in the MoE's own final epilogue
// (k_down, k_grouped_combine), so it costs no launch.
//
// The hidden state of a token holds hc streams of H values (n = hc * H).
// qwen4_verifier.py:20-33 (_hyper) and patch_rmsnorm.py:108-135 (_rms_norm):
//
//   normed  = rms_norm(hidden)              mean of squares per group of gs
//                                           (gs = n: the whole row), fp32
//   d       = silu(W_down . normed / hc)    [lowrank], Q4/G32 vector form
//   mix     = sigmoid(W_up . d)             [n]
//   mixed   = mean_j(mix_j * normed_j)      [H], the branch input
//   weights = 2 * sigmoid(W_inj . normed / hc)   [hc]
//
// every step rounded to the activation type as MLX's bf16 arrays are.
//
//   k_hc_front  per token, blocks of four waves: the block normalises the
//               row into LDS (deterministic chunk sums of 64 squares, then one
//               wave sum per group), block 0 writes `normed`; each wave then
//               computes one row of W_down or W_inj against it.  The row's
//               weights, the streams and the gain are all loaded at entry.
//   k_hc_up     per token, a thread per output element h: the hc rows
//               j * H + h of W_up against d (staged in LDS), the sigmoid, the
//               products with the normalised streams and their mean; the
//               rows' first groups and the stream values load before d.
//
// bf16 calls of kHcTileMin stream values and more run tiles of 16 tokens on the
// matrix cores instead (k_hc_inv, k_hc_low, k_hc_mix below): per token the two
// kernels above read and unpack every projection again (n = 10240, 700
// tokens: 86 + 40 us).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "vm_internal.h"

namespace vm {

namespace {

constexpr int kHcThreads = 256;
constexpr int kHcWaves = kHcThreads / 64;

// Lanes without data load from here: every load is unconditional (a select
// of the address), so the loads issue back to back; a conditional load
// becomes a branch with a wait after it.
__device__ uint4 g_hc_zero[2];

__device__ __forceinline__ const void* or_zero(const void* p, bool live) {
  return live ? p : static_cast<const void*>(g_hc_zero);
}

// Eight consecutive activations (one 16-byte load in bf16, two in fp32),
// kept as raw bits until used.
template <class A>
struct Unit8 {
  uint4 a, b;
  __device__ __forceinline__ void load(const void* p, size_t i, bool live) {
    if constexpr (A::kBytes == 2) {
      a = ldg16(or_zero(static_cast<const uint16_t*>(p) + i, live));
    } else {
      a = ldg16(or_zero(static_cast<const float*>(p) + i, live));
      b = ldg16(or_zero(static_cast<const float*>(p) + i + 4, live));
    }
  }
  __device__ __forceinline__ float get(int k) const {
    if constexpr (A::kBytes == 2) {
      const uint32_t w = k < 2 ? a.x : k < 4 ? a.y : k < 6 ? a.z : a.w;
      return bf16_to_f32(k & 1 ? w >> 16 : w & 0xffffu);
    } else {
      const uint4& q = k < 4 ? a : b;
      const uint32_t w = (k & 3) == 0 ? q.x : (k & 3) == 1 ? q.y : (k & 3) == 2 ? q.z : q.w;
      return __uint_as_float(w);
    }
  }
};

template <class A>
__device__ __forceinline__ void store8(void* p, size_t i, const float y[8]) {
  if constexpr (A::kBytes == 2) {
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = f32_to_bf16(y[2 * k]) | (f32_to_bf16(y[2 * k + 1]) << 16);
    *reinterpret_cast<uint4*>(static_cast<uint16_t*>(p) + i) = make_uint4(w[0], w[1], w[2], w[3]);
  } else {
    float4* q = reinterpret_cast<float4*>(static_cast<float*>(p) + i);
    q[0] = make_float4(y[0], y[1], y[2], y[3]);
    q[1] = make_float4(y[4], y[5], y[6], y[7]);
  }
}

// One Q4/G32 group in the vector form: s * sum(x * q) + b * sum(x).
__device__ __forceinline__ float q4_group(const uint4 words, float s, float b, const float* x) {
#pragma clang fp contract(off)
  const uint32_t w[4] = {words.x, words.y, words.z, words.w};
  float xq = 0.0f, xs = 0.0f;
#pragma unroll
  for (int k = 0; k < kGroup; ++k) {
    const float q = static_cast<float>((w[k / 8] >> (4 * (k % 8))) & 15u);
    xq = xq + x[k] * q;
    xs = xs + x[k];
  }
  return s * xq + b * xs;
}

constexpr int kHcUnits = kHcMaxRow / 8 / kHcThreads;     // 8-element units per thread
constexpr int kHcRowGroups = kHcMaxRow / kGroup / 64;    // Q4 groups of a projection row per lane

template <class A>
__global__ __launch_bounds__(kHcThreads) void k_hc_front(HcLaunch p) {
#pragma clang fp contract(off)
  // the normalised row, one pad float after every 32: lane l reads group
  // g = l + 64 i from s_x[33 g ...], a different bank for every lane
  __shared__ float s_x[kHcMaxRow + kHcMaxRow / kGroup];
  __shared__ float s_chunk[kHcMaxRow / 64];
  __shared__ float s_inv[kHcMaxRow / 64];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t t = blockIdx.y, n = p.n, gs = p.norm_group, r = p.lowrank, hc = p.hc;
  const size_t row_off = static_cast<size_t>(t) * n;
  const uint32_t units = n / 8, groups = n / kGroup;

  // 0. every load that does not depend on the norm, issued together: this
  //    wave's projection row (W_down rows 0..r-1, then W_inj rows), this
  //    thread's units of the streams and of the gain
  const uint32_t row = blockIdx.x * kHcWaves + wave;
  const bool live_row = row < r + hc;
  const bool down = row < r;
  const ProjPtrs pj = down ? p.down : p.inj;
  const uint32_t pr = down ? row : row - r;
  uint4 wq[kHcRowGroups];
  uint32_t wsb[kHcRowGroups], wbb[kHcRowGroups];
#pragma unroll
  for (int i = 0; i < kHcRowGroups; ++i) {
    const uint32_t g = lane + 64u * i;
    const bool live = live_row && g < groups;
    const size_t gi = static_cast<size_t>(pr) * groups + g;
    wq[i] = ldg16(or_zero(pj.w + gi * kWordsPerGroup, live));
    wsb[i] = ldg_u16(or_zero(pj.s + gi, live));
    wbb[i] = ldg_u16(or_zero(pj.b + gi, live));
  }
  Unit8<A> xu[kHcUnits], gu[kHcUnits];
#pragma unroll
  for (int i = 0; i < kHcUnits; ++i) {
    const uint32_t u = tid + kHcThreads * i;
    xu[i].load(p.hidden, row_off + 8 * u, u < units);
    gu[i].load(p.norm_weight, 8 * u, u < units);
  }

  // 1. sums of squares of every 64-element chunk (lanes 8c..8c+7 of a wave
  //    hold chunk c's eight units); n % 64 == 0 keeps those lanes together
#pragma unroll
  for (int i = 0; i < kHcUnits; ++i) {
    const uint32_t u = tid + kHcThreads * i;
    if (u >= units) break;  // uniform over each group of 8 lanes
    float sq = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) sq = sq + xu[i].get(k) * xu[i].get(k);
    sq = group_sum<8>(sq);
    if ((u & 7u) == 7u) s_chunk[u / 8] = sq;
  }
  lds_barrier();

  // 2. 1 / sqrt(mean + eps) of every group, one wave per group
  const uint32_t cpg = gs / 64;
  for (uint32_t g = wave; g < n / gs; g += kHcWaves) {
    float s = 0.0f;
    for (uint32_t c = lane; c < cpg; c += 64) s = s + s_chunk[g * cpg + c];
    s = wave_sum_all(s);
    if (lane == 0) s_inv[g] = 1.0f / sqrtf(s / static_cast<float>(gs) + p.eps);
  }
  lds_barrier();

  // 3. normalise: (x * inv) * gain, rounded to the activation type, into LDS
  //    (and block 0 of the token writes `normed`)
#pragma unroll
  for (int i = 0; i < kHcUnits; ++i) {
    const uint32_t u = tid + kHcThreads * i;
    if (u >= units) break;
    const float inv = s_inv[8 * u / gs];
    float y[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float w = gu[i].get(k);
      const float gain = p.one_centered ? w : 1.0f + w;
      y[k] = A::round((xu[i].get(k) * inv) * gain);
      s_x[8 * u + k + u / 4] = y[k];  // element e at e + e / 32
    }
    if (blockIdx.x == 0) store8<A>(p.normed, row_off + 8 * u, y);
  }
  lds_barrier();

  // 4. the wave's projection row against the normalised row
  if (!live_row) return;
  float acc = 0.0f;
#pragma unroll
  for (int i = 0; i < kHcRowGroups; ++i) {
    const uint32_t g = lane + 64u * i;
    if (g < groups) acc = acc + q4_group(wq[i], bf16_to_f32(wsb[i]), bf16_to_f32(wbb[i]), s_x + g * (kGroup + 1));
  }
  acc = wave_sum_all(acc);
  if (lane != 0) return;
  const float a = A::round(A::round(acc) / static_cast<float>(hc));
  if (down) {
    A::store(p.d, static_cast<size_t>(t) * r + row, A::round(a * sigmoid_act<A>(a)));
  } else {
    A::store(p.weights, static_cast<size_t>(t) * hc + pr, A::round(2.0f * sigmoid_act<A>(a)));
  }
}

template <class A>
__global__ __launch_bounds__(kHcThreads) void k_hc_up(HcLaunch p) {
#pragma clang fp contract(off)
  __shared__ float s_d[kHcMaxLowrank];
  const uint32_t t = blockIdx.y, r = p.lowrank, hc = p.hc, H = p.width;
  const uint32_t h = blockIdx.x * kHcThreads + threadIdx.x;
  const bool live = h < H;
  const uint32_t groups = r / kGroup;
  // the first group of every stream's W_up row and the normalised stream
  // values, issued before the wait for d
  uint4 w0[kMaxStreams];
  uint32_t s0[kMaxStreams], b0[kMaxStreams], xn[kMaxStreams];
#pragma unroll
  for (int j = 0; j < static_cast<int>(kMaxStreams); ++j) {
    const bool lj = live && static_cast<uint32_t>(j) < hc;
    const size_t gi = (static_cast<size_t>(j) * H + h) * groups;
    w0[j] = ldg16(or_zero(p.up.w + gi * kWordsPerGroup, lj));
    s0[j] = ldg_u16(or_zero(p.up.s + gi, lj));
    b0[j] = ldg_u16(or_zero(p.up.b + gi, lj));
    const size_t xi = static_cast<size_t>(t) * p.n + j * H + h;
    xn[j] = A::kBytes == 2 ? ldg_u16(or_zero(static_cast<const uint16_t*>(p.normed) + xi, lj))
                           : ldg_u32(or_zero(static_cast<const float*>(p.normed) + xi, lj));
  }
  for (uint32_t k = threadIdx.x; k < r; k += kHcThreads) s_d[k] = A::load(p.d, static_cast<size_t>(t) * r + k);
  __syncthreads();
  if (!live) return;
  float total = 0.0f;
#pragma unroll
  for (int j = 0; j < static_cast<int>(kMaxStreams); ++j) {
    if (static_cast<uint32_t>(j) >= hc) break;
    const size_t gi = (static_cast<size_t>(j) * H + h) * groups;
    float acc = q4_group(w0[j], bf16_to_f32(s0[j]), bf16_to_f32(b0[j]), s_d);
    for (uint32_t g = 1; g < groups; ++g)
      acc = acc + q4_group(ldg16(p.up.w + (gi + g) * kWordsPerGroup), bf16_to_f32(ldg_u16(p.up.s + gi + g)),
                           bf16_to_f32(ldg_u16(p.up.b + gi + g)), s_d + g * kGroup);
    const float mix = sigmoid_act<A>(A::round(acc));
    total = total + A::round(mix * A::from_bits(xn[j]));
  }
  A::store(p.mixed, static_cast<size_t>(t) * H + h, A::round(A::round(total) * A::round(1.0f / static_cast<float>(hc))));
}

// ------------------------------------------------------- 16-token tiles ---
//
//   k_hc_inv  one block per token: 1 / sqrt(mean + eps) of its norm groups, in
//             the order of k_hc_front's sums.
//   k_hc_low  per 16 tokens and K slice of 32 groups (eight per wave):
//             normalises the slice into MFMA A rows (and writes `normed`) and
//             multiplies it with 48 rows of W_down and W_inj.  One
//             16x16x32 MFMA is one Q4 group: the nibbles go in as the exact
//             integers 0..15 in bf16 and the fp32 result is scaled outside,
//             s * sum(x * q) + b * sum(x), the sum of x from an MFMA with
//             ones.  So no weight is rounded and all sums stay fp32, as in the
//             vector form.  The K slices' partial sums go through scratch:
//             with K whole only tokens / 16 blocks would run (44 of 256 CUs
//             at 700 tokens).
//   k_hc_mix  per 16 tokens and 128 outputs: sums the slices of d (and of the
//             injection weights), then each wave computes 32 outputs of every
//             stream, W_up rows as MFMA A rows in the order that leaves a lane
//             eight consecutive outputs of one token.
//
// n = 10240, 700 tokens: 112 us per call per token, 35.7 in tiles (back to back;
// 4096 tokens 595 and 119).  What is left is latency and VALU: about 30
// instructions, two of them transcendental, for each of the 7.2 M mix values.
constexpr int kTileTok = 16;
constexpr int kLowBlocks = 3;                 // 16-row blocks of projection rows per block
constexpr int kLowRows = 16 * kLowBlocks;
constexpr int kLowGroups = 8;                 // Q4 groups per wave: one 16-byte load of scales per row

__host__ __device__ constexpr uint32_t low_slices(uint32_t n) {
  return (n / kGroup + kHcWaves * kLowGroups - 1) / (kHcWaves * kLowGroups);
}
constexpr uint32_t kMaxSlices = low_slices(kHcMaxRow);
__host__ __device__ constexpr uint32_t low_row_blocks(uint32_t rows) { return (rows + kLowRows - 1) / kLowRows; }

typedef __bf16 hc_bf16x8 __attribute__((ext_vector_type(8)));
typedef float hc_f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ hc_f32x4 hc_mfma(const uint4 a, const uint4 b) {
  const hc_f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(hc_bf16x8, a), __builtin_bit_cast(hc_bf16x8, b),
                                                 zero, 0, 0, 0);
}

// The eight nibbles of a word as bf16 integers, in input order.
__device__ __forceinline__ uint4 nibbles_bf16(uint32_t w) {
  const uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;  // bytes: even and odd nibbles
  uint32_t out[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = static_cast<float>((lo >> (8 * i)) & 0xffu), b = static_cast<float>((hi >> (8 * i)) & 0xffu);
    out[i] = (__float_as_uint(a) >> 16) | __float_as_uint(b);  // integers up to 15: the low halves are zero
  }
  return make_uint4(out[0], out[1], out[2], out[3]);
}

__device__ __forceinline__ uint32_t half16(const uint4 v, int k) {
  const uint32_t w = k < 2 ? v.x : k < 4 ? v.y : k < 6 ? v.z : v.w;
  return k & 1 ? w >> 16 : w & 0xffffu;
}

__device__ __forceinline__ float* tile_inv(const HcLaunch& p) {
  const uint32_t tiles = (p.tokens + kTileTok - 1) / kTileTok;
  return p.tile_ws +
         static_cast<size_t>(tiles) * low_slices(p.n) * low_row_blocks(p.lowrank + p.hc) * kLowRows * kTileTok;
}

__global__ __launch_bounds__(kHcThreads) void k_hc_inv(HcLaunch p) {
#pragma clang fp contract(off)
  __shared__ float s_chunk[kHcMaxRow / 64];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t t = blockIdx.x, n = p.n, gs = p.norm_group, units = n / 8;
  const size_t row_off = static_cast<size_t>(t) * n;
  Unit8<ActBF16> xu[kHcUnits];
#pragma unroll
  for (int i = 0; i < kHcUnits; ++i) {
    const uint32_t u = tid + kHcThreads * i;
    xu[i].load(p.hidden, row_off + 8 * u, u < units);
  }
#pragma unroll
  for (int i = 0; i < kHcUnits; ++i) {
    const uint32_t u = tid + kHcThreads * i;
    if (u >= units) break;
    float sq = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) sq = sq + xu[i].get(k) * xu[i].get(k);
    sq = group_sum<8>(sq);
    if ((u & 7u) == 7u) s_chunk[u / 8] = sq;
  }
  lds_barrier();
  const uint32_t cpg = gs / 64;
  float* inv = tile_inv(p) + static_cast<size_t>(t) * (n / gs);
  for (uint32_t g = wave; g < n / gs; g += kHcWaves) {
    float s = 0.0f;
    for (uint32_t c = lane; c < cpg; c += 64) s = s + s_chunk[g * cpg + c];
    s = wave_sum_all(s);
    if (lane == 0) inv[g] = 1.0f / sqrtf(s / static_cast<float>(gs) + p.eps);
  }
}

__global__ __launch_bounds__(kHcThreads, 3) void k_hc_low(HcLaunch p) {
  __shared__ __align__(16) float s_part[kHcWaves][kLowRows * (kTileTok + 4)];  // row * 20 + token
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lc = lane & 15u, kb = lane >> 4;
  const uint32_t n = p.n, groups = n / kGroup, r = p.lowrank, rows = r + p.hc;
  const uint32_t t0 = blockIdx.y * kTileTok, row0 = blockIdx.z * kLowRows;
  const uint32_t g0 = (blockIdx.x * kHcWaves + wave) * kLowGroups;
  const uint32_t token = min(t0 + lc, p.tokens - 1);  // rows past the end repeat the last token
  hc_f32x4 acc[kLowBlocks];
#pragma unroll
  for (int b = 0; b < kLowBlocks; ++b) acc[b] = hc_f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  if (g0 < groups) {  // wave-uniform; n % 256 == 0, so the eight groups are all inside the row
    const uint16_t* xrow = static_cast<const uint16_t*>(p.hidden) + static_cast<size_t>(token) * n + g0 * kGroup + kb * 8;
    const uint16_t* grow = static_cast<const uint16_t*>(p.norm_weight) + g0 * kGroup + kb * 8;
    const uint32_t* wrow[kLowBlocks];
    uint4 sv[kLowBlocks], bv[kLowBlocks];
#pragma unroll
    for (int b = 0; b < kLowBlocks; ++b) {
      const uint32_t row = min(row0 + 16u * b + lc, rows - 1);  // repeated rows are not stored
      const ProjPtrs& pj = row < r ? p.down : p.inj;
      const size_t at = static_cast<size_t>(row < r ? row : row - r) * groups + g0;
      wrow[b] = pj.w + at * kWordsPerGroup + kb;
      sv[b] = ldg16(pj.s + at);
      bv[b] = ldg16(pj.b + at);
    }
    // norm group of the first Q4 group, and the inputs of it that lie before
    uint32_t norm = g0 * kGroup / p.norm_group, past = g0 * kGroup % p.norm_group;
    const float* inv = tile_inv(p) + static_cast<size_t>(token) * (n / p.norm_group);
    uint4 xv[kLowGroups], gv[kLowGroups];
    uint32_t wv[kLowGroups][kLowBlocks];
    float iv[kLowGroups];
#pragma unroll
    for (int i = 0; i < kLowGroups; ++i) {
      xv[i] = ldg16(xrow + i * kGroup);
      gv[i] = ldg16(grow + i * kGroup);
      iv[i] = inv[norm];
      past += kGroup;
      if (past == p.norm_group) {
        past = 0;
        ++norm;
      }
#pragma unroll
      for (int b = 0; b < kLowBlocks; ++b) wv[i][b] = ldg_u32(wrow[b] + i * kWordsPerGroup);
    }
    const uint4 ones = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
    const bool write = blockIdx.z == 0 && t0 + lc < p.tokens;
    uint16_t* nrow = static_cast<uint16_t*>(p.normed) + static_cast<size_t>(token) * n + g0 * kGroup + kb * 8;
#pragma unroll
    for (int i = 0; i < kLowGroups; ++i) {
      uint32_t y[8];
      {
#pragma clang fp contract(off)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float w = bf16_to_f32(half16(gv[i], k));
          const float gain = p.one_centered ? w : 1.0f + w;
          y[k] = f32_to_bf16((bf16_to_f32(half16(xv[i], k)) * iv[i]) * gain);
        }
      }
      const uint4 a = make_uint4(y[0] | y[1] << 16, y[2] | y[3] << 16, y[4] | y[5] << 16, y[6] | y[7] << 16);
      if (write) *reinterpret_cast<uint4*>(nrow + i * kGroup) = a;
      const hc_f32x4 xs = hc_mfma(a, ones);
#pragma unroll
      for (int b = 0; b < kLowBlocks; ++b) {
        const hc_f32x4 xq = hc_mfma(a, nibbles_bf16(wv[i][b]));
        const float s = bf16_to_f32(half16(sv[b], i)), bi = bf16_to_f32(half16(bv[b], i));
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[b][e] += fmaf(s, xq[e], bi * xs[e]);
      }
    }
  }
  // lane: tokens 4 kb .. 4 kb + 3 of row 16 b + lc
#pragma unroll
  for (int b = 0; b < kLowBlocks; ++b)
    *reinterpret_cast<hc_f32x4*>(&s_part[wave][(16 * b + lc) * (kTileTok + 4) + 4 * kb]) = acc[b];
  __syncthreads();
  float* out = p.tile_ws + ((static_cast<size_t>(blockIdx.y) * gridDim.x + blockIdx.x) * gridDim.z + blockIdx.z) *
                               (kLowRows * kTileTok);
#pragma unroll
  for (uint32_t idx = tid; idx < kLowRows * kTileTok; idx += kHcThreads) {
    const uint32_t at = (idx / kTileTok) * (kTileTok + 4) + idx % kTileTok;
    float v = s_part[0][at];
#pragma unroll
    for (int w = 1; w < kHcWaves; ++w) v += s_part[w][at];
    out[idx] = v;
  }
}

// ONE: lowrank 32, one group per W_up row, whose scales are then contiguous
// over the rows.
// HC: bound of the stream count (registers for the streams' loads).
template <bool ONE, int HC>
__global__ __launch_bounds__(kHcThreads, HC > 4 ? 3 : 4) void k_hc_mix(HcLaunch p) {
  constexpr int kStride = kHcMaxLowrank + 8;  // bf16 per token of d, 16 bytes of padding
  __shared__ __align__(16) uint16_t s_d[kTileTok * kStride];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lc = lane & 15u, kb = lane >> 4;
  const uint32_t n = p.n, H = p.width, r = p.lowrank, hc = p.hc, rg = r / kGroup;
  const uint32_t t0 = blockIdx.y * kTileTok;
  const uint32_t token = min(t0 + lc, p.tokens - 1);
  const uint32_t hg = blockIdx.x * kHcWaves + wave;
  const bool live = hg * kGroup < H;
  const uint32_t h0 = live ? hg * kGroup : 0;
  // W_up row of A row lc of half m: the lane's C rows 4 kb + i are then the
  // outputs h0 + 8 kb + 4 m + i
  const uint32_t arow = (lc >> 2) * 8 + (lc & 3u);
  const uint16_t* xrow = static_cast<const uint16_t*>(p.normed) + static_cast<size_t>(token) * n + h0 + kb * 8;

  uint4 xv[HC], sv[HC], bv[HC];
  uint32_t wv[HC][2];
#pragma unroll
  for (int j = 0; j < HC; ++j) {
    if (static_cast<uint32_t>(j) >= hc) break;
    const size_t o0 = static_cast<size_t>(j) * H + h0;
    xv[j] = ldg16(xrow + static_cast<size_t>(j) * H);
    if constexpr (ONE) {
      sv[j] = ldg16(p.up.s + o0 + kb * 8);
      bv[j] = ldg16(p.up.b + o0 + kb * 8);
#pragma unroll
      for (int m = 0; m < 2; ++m) wv[j][m] = ldg_u32(p.up.w + (o0 + arow + 4 * m) * kWordsPerGroup + kb);
    }
  }

  // d of the tile's tokens, and in the first blocks the injection weights
  const uint32_t slices = low_slices(n), padded = low_row_blocks(r + hc) * kLowRows;
  const float* part = p.tile_ws + static_cast<size_t>(blockIdx.y) * slices * padded * kTileTok;
  const uint32_t want = (blockIdx.x == 0 ? r + hc : r) * kTileTok;
  for (uint32_t idx = tid; idx < want; idx += kHcThreads) {
    const uint32_t row = idx / kTileTok, tok = idx % kTileTok;
    float v[kMaxSlices], sum = 0.0f;  // all slices' loads go out together
#pragma unroll
    for (uint32_t k = 0; k < kMaxSlices; ++k) v[k] = part[min(k, slices - 1) * padded * kTileTok + idx];
#pragma unroll
    for (uint32_t k = 0; k < kMaxSlices; ++k) sum += k < slices ? v[k] : 0.0f;
    const float a = round_bf16(round_bf16(sum) / static_cast<float>(hc));
    const float sig = sigmoid_act<ActBF16>(a);
    const bool store = blockIdx.x == 0 && t0 + tok < p.tokens;
    if (row < r) {
      const uint16_t d = static_cast<uint16_t>(f32_to_bf16(a * sig));
      s_d[tok * kStride + row] = d;
      if (store) static_cast<uint16_t*>(p.d)[static_cast<size_t>(t0 + tok) * r + row] = d;
    } else if (store) {
      ActBF16::store(p.weights, static_cast<size_t>(t0 + tok) * hc + (row - r), round_bf16(2.0f * sig));
    }
  }
  __syncthreads();
  if (!live) return;

  const uint4 ones = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
  const auto d_of = [&](uint32_t g) { return *reinterpret_cast<const uint4*>(&s_d[lc * kStride + g * kGroup + kb * 8]); };
  const uint4 d0 = d_of(0);
  const float ds0 = hc_mfma(ones, d0)[0];
  float total[8] = {};
#pragma unroll
  for (int j = 0; j < HC; ++j) {
    if (static_cast<uint32_t>(j) >= hc) break;
    float acc[8];
    if constexpr (ONE) {
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const hc_f32x4 dq = hc_mfma(nibbles_bf16(wv[j][m]), d0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[4 * m + i] = fmaf(bf16_to_f32(half16(sv[j], 4 * m + i)), dq[i], bf16_to_f32(half16(bv[j], 4 * m + i)) * ds0);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
      const size_t o0 = static_cast<size_t>(j) * H + h0;
      for (uint32_t g = 0; g < rg; ++g) {
        const uint4 dg = d_of(g);
        const float ds = hc_mfma(ones, dg)[0];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const hc_f32x4 dq = hc_mfma(nibbles_bf16(ldg_u32(p.up.w + ((o0 + arow + 4 * m) * rg + g) * kWordsPerGroup + kb)), dg);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const size_t at = (o0 + kb * 8 + 4 * m + i) * rg + g;
            acc[4 * m + i] += fmaf(bf16_to_f32(ldg_u16(p.up.s + at)), dq[i], bf16_to_f32(ldg_u16(p.up.b + at)) * ds);
          }
        }
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma clang fp contract(off)
      const float mix = sigmoid_act<ActBF16>(round_bf16(acc[e]));
      total[e] = total[e] + round_bf16(mix * bf16_to_f32(half16(xv[j], e)));
    }
  }
  if (t0 + lc >= p.tokens) return;
  const float scale = round_bf16(1.0f / static_cast<float>(hc));
  uint32_t y[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = f32_to_bf16(round_bf16(total[e]) * scale);
  *reinterpret_cast<uint4*>(static_cast<uint16_t*>(p.mixed) + static_cast<size_t>(token) * H + h0 + kb * 8) =
      make_uint4(y[0] | y[1] << 16, y[2] | y[3] << 16, y[4] | y[5] << 16, y[6] | y[7] << 16);
}

template <class K>
hipError_t launch_timed(const char* family, K kernel, dim3 grid, const HcLaunch& p, hipStream_t stream) {
  hipEvent_t start = nullptr, stop = nullptr;
  if (timing_events(family, &start, &stop))
    hipExtLaunchKernelGGL(kernel, grid, dim3(kHcThreads), 0, stream, start, stop, 0, p);
  else
    hipLaunchKernelGGL(kernel, grid, dim3(kHcThreads), 0, stream, p);
  return hipGetLastError();
}

}  // namespace

uint64_t hyper_tile_bytes(uint32_t tokens, uint32_t n, uint32_t rows) {
  const uint64_t tiles = (tokens + kTileTok - 1) / kTileTok;
  return tiles * low_slices(n) * low_row_blocks(rows) * kLowRows * kTileTok * 4 + uint64_t(tokens) * (n / 64) * 4;
}

bool hyper_tiled(const HcLaunch& p) {
  const auto aligned = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15u) == 0; };
  return p.act_dtype == 0 && static_cast<uint64_t>(p.tokens) * p.n >= kHcTileMin && p.width % kGroup == 0 && p.n % (8 * kGroup) == 0 &&
         aligned(p.mixed) && aligned(p.down.s) && aligned(p.down.b) && aligned(p.inj.s) && aligned(p.inj.b) &&
         aligned(p.up.s) && aligned(p.up.b);
}

hipError_t launch_hyper_mix(const HcLaunch& p, hipStream_t stream) {
  if (p.tile_ws != nullptr && hyper_tiled(p)) {
    const uint32_t tiles = (p.tokens + kTileTok - 1) / kTileTok;
    hipError_t e = launch_timed("hc_inv", k_hc_inv, dim3(p.tokens), p, stream);
    if (e != hipSuccess) return e;
    e = launch_timed("hc_low", k_hc_low, dim3(low_slices(p.n), tiles, low_row_blocks(p.lowrank + p.hc)), p, stream);
    if (e != hipSuccess) return e;
    const dim3 mix((p.width / kGroup + kHcWaves - 1) / kHcWaves, tiles);
    if (p.lowrank != kGroup) return launch_timed("hc_mix", k_hc_mix<false, kMaxStreams>, mix, p, stream);
    return p.hc <= 4 ? launch_timed("hc_mix", k_hc_mix<true, 4>, mix, p, stream)
                     : launch_timed("hc_mix", k_hc_mix<true, kMaxStreams>, mix, p, stream);
  }
  const dim3 front((p.lowrank + p.hc + kHcWaves - 1) / kHcWaves, p.tokens);
  const dim3 up((p.width + kHcThreads - 1) / kHcThreads, p.tokens);
  hipError_t e = p.act_dtype == 0 ? launch_timed("hc_front", k_hc_front<ActBF16>, front, p, stream)
                                  : launch_timed("hc_front", k_hc_front<ActF32>, front, p, stream);
  if (e != hipSuccess) return e;
  return p.act_dtype == 0 ? launch_timed("hc_up", k_hc_up<ActBF16>, up, p, stream)
                          : launch_timed("hc_up", k_hc_up<ActF32>, up, p, stream);
}

}  // namespace vm
