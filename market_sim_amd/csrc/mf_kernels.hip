// gfx950 kernels of the reference operators: RMSNorm, the fixed-width
// restricted output head (restricted_output_head_f16), the selections over
// precomputed logits and the small-shape linear_f16.  The decode tail lives
// in mf_tail.hip.
//
// Build: hipcc --offload-arch=gfx950 -ffp-contract=off (see csrc/Makefile).
// -ffp-contract=off keeps every reference-order multiply-add unfused unless
// written as an explicit fma.
#include <hip/hip_runtime.h>

#include "mf_device.hpp"
#include "mf_launch.hpp"
#include "mf_norm.hpp"

namespace mf {
namespace {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;

// ---------------------------------------------------------------------------
// Final RMSNorm in the reference FP32 CPU order (src/cpu/operators.cpp:
// 523-535): one wave per row; lane 0 runs the sequential unfused sum of
// squares over the row staged in LDS, then every lane writes
// (x * inverse) * weight.  Optionally writes an upper bound of ||y||_2 per
// row for the MFMA bounds.
// ---------------------------------------------------------------------------
// Rows up to this width also stage the weight in LDS (3 H floats in all).
constexpr uint32_t kNormStagedWeightMax = 8192;

template <bool kHalfIn, bool kHalfW, bool kHalfOut>
__global__ __launch_bounds__(kWave) void rms_norm_kernel(
    const void* __restrict__ input, const void* __restrict__ weight,
    void* output, float* __restrict__ row_norm, uint32_t H, float epsilon) {
  // [H] x, [H] x * x, and [H] weight when H <= kNormStagedWeightMax
  extern __shared__ __align__(16) float xs[];
  __shared__ float inverse_shared;
  const bool stage_w = H <= kNormStagedWeightMax;
  float* sq = xs + H;
  float* ws = xs + 2u * H;
  const uint64_t r = blockIdx.x;
  const uint32_t lane = threadIdx.x;
  // x and the weight staged with four 4-element loads of each per lane in
  // flight before the LDS stores (one memory round trip per 1024 features)
  constexpr uint32_t kInBytes = kHalfIn ? 2u : 4u;
  constexpr uint32_t kWBytes = kHalfW ? 2u : 4u;
  const bool vec = (H & 3u) == 0 &&
                   (reinterpret_cast<uintptr_t>(input) & (4u * kInBytes - 1u)) == 0 &&
                   (reinterpret_cast<uintptr_t>(weight) & (4u * kWBytes - 1u)) == 0;
  auto load4 = [](const void* base, uint64_t q, auto half) -> float4 {
    if constexpr (decltype(half)::value) {
      const uint2 h = static_cast<const uint2*>(base)[q];
      return float4{half_to_float(static_cast<uint16_t>(h.x)), half_to_float(static_cast<uint16_t>(h.x >> 16)),
                    half_to_float(static_cast<uint16_t>(h.y)), half_to_float(static_cast<uint16_t>(h.y >> 16))};
    } else {
      return static_cast<const float4*>(base)[q];
    }
  };
  using HalfIn = std::integral_constant<bool, kHalfIn>;
  using HalfW = std::integral_constant<bool, kHalfW>;
  if (vec) {
    constexpr uint32_t kBatch = 4;
    const uint32_t n4 = H / 4u;
    for (uint32_t base = lane; base < n4; base += kWave * kBatch) {
      float4 v[kBatch];
      float4 w4[kBatch];
#pragma unroll
      for (uint32_t u = 0; u < kBatch; ++u) {
        const uint32_t q = base + u * kWave;
        v[u] = q < n4 ? load4(input, r * n4 + q, HalfIn{}) : float4{0.0f, 0.0f, 0.0f, 0.0f};
        w4[u] = (stage_w && q < n4) ? load4(weight, q, HalfW{}) : float4{0.0f, 0.0f, 0.0f, 0.0f};
      }
#pragma unroll
      for (uint32_t u = 0; u < kBatch; ++u) {
        const uint32_t q = base + u * kWave;
        if (q < n4) {
          reinterpret_cast<float4*>(xs)[q] = v[u];
          reinterpret_cast<float4*>(sq)[q] =
              float4{v[u].x * v[u].x, v[u].y * v[u].y, v[u].z * v[u].z, v[u].w * v[u].w};
          if (stage_w) reinterpret_cast<float4*>(ws)[q] = w4[u];
        }
      }
    }
  } else {
    for (uint32_t c = lane; c < H; c += kWave) {
      const float v = kHalfIn ? half_to_float(static_cast<const uint16_t*>(input)[r * H + c])
                              : static_cast<const float*>(input)[r * H + c];
      xs[c] = v;
      sq[c] = v * v;
      if (stage_w) {
        ws[c] = kHalfW ? half_to_float(static_cast<const uint16_t*>(weight)[c])
                       : static_cast<const float*>(weight)[c];
      }
    }
  }
  __syncthreads();
  // sum of the squares in feature order, then mean, + epsilon, sqrt and
  // reciprocal, each rounded once (rms_norm.cu:104-182)
  const float sum_squares = sequential_sum_wave(sq, H);
  if (lane == 0) inverse_shared = norm_inverse(sum_squares, H, epsilon);
  __syncthreads();
  const float inverse = inverse_shared;
  float norm_sq = 0.0f;
  for (uint32_t c = lane; c < H; c += kWave) {
    const float w = stage_w ? ws[c]
                    : kHalfW ? half_to_float(static_cast<const uint16_t*>(weight)[c])
                             : static_cast<const float*>(weight)[c];
    const float scaled = xs[c] * inverse;
    const float y = scaled * w;
    if constexpr (kHalfOut) {
      static_cast<uint16_t*>(output)[r * H + c] = float_to_half_rne(y);
    } else {
      static_cast<float*>(output)[r * H + c] = y;
      norm_sq = __builtin_fmaf(y, y, norm_sq);
    }
  }
  if (row_norm != nullptr) {
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) {
      norm_sq += __shfl_xor(norm_sq, m);
    }
    if (lane == 0) {
      // The FP32 sum of H squares is within a relative H * 2^-24 of the exact
      // value; the factor below covers that and the sqrt rounding for any
      // H <= 2^16.
      row_norm[r] = __fsqrt_rn(norm_sq) * (1.0f + 0x1p-7f);
    }
  }
}

// The same norm for many rows: a wave takes 64 / G rows, G lanes a row
// (split by norm_split).  Lane k of a row holds segment k of it, S
// 16-byte words, in registers; the running sums go through the segments in
// order, handed one lane up (DPP) after each, so every row of the wave is in
// its chain at once and the additions and their order are the reference's.
// An FP16 square is exact in FP32, so fma(x, x, s) is the reference's rounded
// square and sum in one instruction on the packed halves.
// The rows are read once, in contiguous words that stay in registers for the
// output; the segments are dealt through LDS (a lane's segment at an odd
// number of 16-byte words, so 16 lanes meet 16 bank groups).
// Bound: with a wave a SIMD or fewer the chain (H dependent additions, about
// 5 cycles each), beyond that the SIMDs' issue of H additions per wave.
// 2048 x 2048 FP16: 25.3 -> 9.4 us a call, FP32 28.5 -> 12.8; 8192 x 4096
// FP16: 300 -> 45 us, FP32 282 -> 73 (3.7 TB/s); 1 x 576: 5.7 -> 5.6 (from one
// row a wave with x, its squares and the weight in LDS, which held six rows of
// 2048 a compute unit; that kernel keeps the rows that are not whole words, or
// wider).
struct NormSplit {
  uint32_t lanes_log2;  // G
  uint32_t per_wave;    // rows per wave, at most 64 / G
  uint32_t words;       // 16-byte words per row
  uint32_t row_magic;   // q / words = q * row_magic >> 20 for q < 1024
};
constexpr uint32_t kNormSegMax = 16;   // words per segment: 4, 8, 12 or 16
constexpr uint32_t kNormWaves = 1024;  // waves (one a SIMD) before waves take more rows

template <bool kHalf, uint32_t kSeg>
__global__ __launch_bounds__(kWave) void rms_norm_rows_kernel(const void* input,
                                                              const void* __restrict__ weight,
                                                              void* output, uint32_t rows,
                                                              uint32_t H, float epsilon,
                                                              NormSplit d) {
  constexpr uint32_t kStride = kSeg | 1u;
  __shared__ uint4 seg_lds[kWave * kStride];
  const uint32_t lane = threadIdx.x;
  const uint32_t first = blockIdx.x * d.per_wave;
  const uint32_t n = (rows - first < d.per_wave ? rows - first : d.per_wave) * d.words;
  const uint4* src = static_cast<const uint4*>(input) + static_cast<uint64_t>(first) * d.words;
  uint4* dst = static_cast<uint4*>(output) + static_cast<uint64_t>(first) * d.words;
  const uint4* wsrc = static_cast<const uint4*>(weight);
  // word lane + 64 i of the wave's rows (past the end: the last word again,
  // read, dealt and written with the same value), at most kSeg per lane
  uint32_t at = lane;
  auto word_at = [&](uint32_t i) {
    const uint32_t q = at + kWave * i;
    return q < n ? q : n - 1u;
  };
  uint4 v[kSeg];
#pragma unroll
  for (uint32_t i = 0; i < kSeg; ++i) v[i] = src[word_at(i)];
#pragma unroll
  for (uint32_t i = 0; i < kSeg; ++i) {
    const uint32_t q = word_at(i);
    const uint32_t j = (q * d.row_magic) >> 20;
    const uint32_t w = q - j * d.words;
    const uint32_t k = w / kSeg;
    seg_lds[((j << d.lanes_log2) + k) * kStride + (w - k * kSeg)] = v[i];
  }
  wave_sync();
  const uint32_t begin = (lane & ((1u << d.lanes_log2) - 1u)) * kSeg;
  const uint32_t have = begin < d.words ? d.words - begin : 0u;
  uint4 sg[kSeg];
#pragma unroll
  for (uint32_t p = 0; p < kSeg; ++p) sg[p] = seg_lds[lane * kStride + p];
#pragma unroll
  for (uint32_t p = 0; p < kSeg; ++p) {
    const uint32_t keep = p < have ? ~0u : 0u;  // past the row: zeros, which add nothing
    sg[p] = uint4{sg[p].x & keep, sg[p].y & keep, sg[p].z & keep, sg[p].w & keep};
    if constexpr (!kHalf) {
      const float f[4] = {as_float(sg[p].x), as_float(sg[p].y), as_float(sg[p].z), as_float(sg[p].w)};
      sg[p] = uint4{as_u32(f[0] * f[0]), as_u32(f[1] * f[1]), as_u32(f[2] * f[2]), as_u32(f[3] * f[3])};
    }
  }
  const uint32_t segments = (d.words + kSeg - 1u) / kSeg;
  // Every lane adds its segment to what it was handed; the lane that holds
  // segment t after t hand-overs holds the row's sum so far.
  float s = 0.0f;
  for (uint32_t t = 0; t < segments; ++t) {
    if (t != 0u) s = lane_shift_right(s);
#pragma unroll
    for (uint32_t p = 0; p < kSeg; ++p) {
      const uint32_t q[4] = {sg[p].x, sg[p].y, sg[p].z, sg[p].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (kHalf) {
          const half2_t h = __builtin_bit_cast(half2_t, q[e]);
          s = __builtin_fmaf(static_cast<float>(h.x), static_cast<float>(h.x), s);
          s = __builtin_fmaf(static_cast<float>(h.y), static_cast<float>(h.y), s);
        } else {
          s = s + as_float(q[e]);
        }
      }
    }
  }
  const float inverse = norm_inverse(s, H, epsilon);  // the row's in lane `segments` - 1 of it
  // the words' places are worked out again: kept over the chain they would
  // cost a register each
  asm volatile("" : "+v"(at));
  constexpr uint32_t kBatch = 4;
#pragma unroll
  for (uint32_t i0 = 0; i0 < kSeg; i0 += kBatch) {
    if (kWave * i0 >= n) break;
    uint4 g[kBatch];
    float inv[kBatch];
#pragma unroll
    for (uint32_t u = 0; u < kBatch; ++u) {
      const uint32_t q = word_at(i0 + u);
      const uint32_t j = (q * d.row_magic) >> 20;
      g[u] = wsrc[q - j * d.words];
      inv[u] = __shfl(inverse, static_cast<int>((j << d.lanes_log2) + segments - 1u));
    }
#pragma unroll
    for (uint32_t u = 0; u < kBatch; ++u) {
      const uint32_t x[4] = {v[i0 + u].x, v[i0 + u].y, v[i0 + u].z, v[i0 + u].w};
      const uint32_t w[4] = {g[u].x, g[u].y, g[u].z, g[u].w};
      uint32_t y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (kHalf) {
          const half2_t a = __builtin_bit_cast(half2_t, x[e]);
          const half2_t b = __builtin_bit_cast(half2_t, w[e]);
          const float y0 = (static_cast<float>(a.x) * inv[u]) * static_cast<float>(b.x);
          const float y1 = (static_cast<float>(a.y) * inv[u]) * static_cast<float>(b.y);
          y[e] = static_cast<uint32_t>(float_to_half_rne(y0)) |
                 (static_cast<uint32_t>(float_to_half_rne(y1)) << 16);
        } else {
          y[e] = as_u32((as_float(x[e]) * inv[u]) * as_float(w[e]));
        }
      }
      dst[word_at(i0 + u)] = uint4{y[0], y[1], y[2], y[3]};
    }
  }
}

// Rows too wide to stage whole in LDS (H > kNormStagedMax): the squares are
// staged kNormChunk features at a time and lane 0 adds them in feature order
// (one running sum across the chunks: the same chain as the staged kernel),
// then y = (x * inverse) * weight with x and the weight read again from
// global memory.
constexpr uint32_t kNormStagedMax = 16384;
constexpr uint32_t kNormChunk = 4096;

template <bool kHalfIn, bool kHalfW, bool kHalfOut>
__global__ __launch_bounds__(kWave) void rms_norm_wide_kernel(
    const void* __restrict__ input, const void* __restrict__ weight,
    void* output, float* __restrict__ row_norm, uint32_t H, float epsilon) {
  __shared__ float sq[kNormChunk];
  __shared__ float inverse_shared;
  const uint64_t r = blockIdx.x;
  const uint32_t lane = threadIdx.x;
  auto x_at = [&](uint64_t c) -> float {
    return kHalfIn ? half_to_float(static_cast<const uint16_t*>(input)[r * H + c])
                   : static_cast<const float*>(input)[r * H + c];
  };
  auto w_at = [&](uint64_t c) -> float {
    return kHalfW ? half_to_float(static_cast<const uint16_t*>(weight)[c])
                  : static_cast<const float*>(weight)[c];
  };
  float sum = 0.0f;  // lane 0's chain
  for (uint32_t base = 0; base < H; base += kNormChunk) {
    const uint32_t n = H - base < kNormChunk ? H - base : kNormChunk;
    for (uint32_t c = lane; c < n; c += kWave) {
      const float v = x_at(base + c);
      sq[c] = v * v;
    }
    __syncthreads();
    if (lane == 0) {
      for (uint32_t c = 0; c < n; ++c) sum = sum + sq[c];
    }
    __syncthreads();
  }
  if (lane == 0) inverse_shared = norm_inverse(sum, H, epsilon);
  __syncthreads();
  const float inverse = inverse_shared;
  float norm_sq = 0.0f;
  for (uint32_t c = lane; c < H; c += kWave) {
    const float y = (x_at(c) * inverse) * w_at(c);
    if constexpr (kHalfOut) {
      static_cast<uint16_t*>(output)[r * H + c] = float_to_half_rne(y);
    } else {
      static_cast<float*>(output)[r * H + c] = y;
      norm_sq = __builtin_fmaf(y, y, norm_sq);
    }
  }
  if (row_norm != nullptr) {
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) norm_sq += __shfl_xor(norm_sq, m);
    if (lane == 0) row_norm[r] = __fsqrt_rn(norm_sq) * (1.0f + 0x1p-7f);
  }
}

// Reference linear_f16 arithmetic on shapes the MFMA tiling does not cover:
// one output per thread, sequential fma over the input features
// (tests/cuda/cuda_tests.cu:170-181 order), rounded to FP16.
__global__ __launch_bounds__(256) void linear_f16_simple_kernel(
    const uint16_t* __restrict__ input, const uint16_t* __restrict__ weight,
    uint16_t* __restrict__ output, uint32_t rows, uint32_t in_features,
    uint32_t out_features) {
  const uint64_t idx = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= static_cast<uint64_t>(rows) * out_features) return;
  const uint64_t r = idx / out_features;
  const uint64_t o = idx % out_features;
  float s = 0.0f;
  for (uint32_t f = 0; f < in_features; ++f) {
    s = __builtin_fmaf(half_to_float(input[r * in_features + f]),
                       half_to_float(weight[o * in_features + f]), s);
  }
  output[idx] = float_to_half_rne(s);
}

// ---------------------------------------------------------------------------
// Restricted head.
// ---------------------------------------------------------------------------

struct RowList {
  const uint32_t* ids;
  uint32_t count;
  int status;  // 0 ok, 1 invalid row
};

// Fixed-width candidate table of the reference restricted head
// (greedy.cu:145-151): count 0 or above the maximum makes the row invalid.
__device__ RowList resolve_row(const HeadArgs& a, uint32_t r) {
  RowList l{nullptr, 0u, 0};
  const uint32_t c = a.fixed_counts[r];
  if (c == 0 || c > a.max_allowed) {
    l.status = 1;
    return l;
  }
  l.ids = a.fixed_ids + static_cast<uint64_t>(r) * a.max_allowed;
  l.count = c;
  return l;
}

// Cross-wave reduction scratch of a workgroup of kW waves.
template <int kW>
struct Red {
  float red_f[kW];
  uint32_t red_u[kW];
  uint32_t red_u2[kW];
  uint32_t red_t[kW];
  uint32_t red_p[kW];
  float red_s[kW];
};

// The head's workgroup: eight waves per row, so that a row of 128 candidates
// of 1152 bytes is in flight at once (one workgroup a compute unit at 256 rows).
constexpr int kHeadThreads = 512;
constexpr int kHeadWaves = kHeadThreads / kWave;

struct HeadShared : Red<kHeadWaves> {
  float sc[kHeadChunkMax];  // fast score g
  float bd[kHeadChunkMax];  // bound b
  uint32_t tk[kHeadChunkMax];
  Record recs[kHeadMaxRecords];
  uint32_t members[kHeadChunkMax];
  uint32_t n_members;
  uint32_t last;
  Record rec;
};

template <int kW>
__device__ __forceinline__ uint32_t block_sum(Red<kW>& sh, uint32_t v) {
  v = wave_sum_u32(v);
  const int w = threadIdx.x / kWave;
  __syncthreads();
  if ((threadIdx.x % kWave) == 0) sh.red_u[w] = v;
  __syncthreads();
  uint32_t out = 0;
#pragma unroll
  for (int i = 0; i < kW; ++i) out += sh.red_u[i];
  return out;
}

template <int kW>
__device__ __forceinline__ Best block_best(Red<kW>& sh, Best b) {
  b = wave_best(b);
  const int w = threadIdx.x / kWave;
  __syncthreads();
  if ((threadIdx.x % kWave) == 0) {
    sh.red_s[w] = b.score;
    sh.red_t[w] = b.token;
    sh.red_p[w] = b.pos;
  }
  __syncthreads();
  Best out{sh.red_s[0], sh.red_t[0], sh.red_p[0]};
#pragma unroll
  for (int i = 1; i < kW; ++i) {
    out = best_of(out, Best{sh.red_s[i], sh.red_t[i], sh.red_p[i]});
  }
  return out;
}

template <int kW>
__device__ __forceinline__ void block_min_token(Red<kW>& sh, uint32_t& t,
                                                uint32_t& p) {
  wave_min_token(t, p);
  const int w = threadIdx.x / kWave;
  __syncthreads();
  if ((threadIdx.x % kWave) == 0) {
    sh.red_u2[w] = t;
    sh.red_p[w] = p;
  }
  __syncthreads();
  t = sh.red_u2[0];
  p = sh.red_p[0];
#pragma unroll
  for (int i = 1; i < kW; ++i) {
    if (sh.red_u2[i] < t) {
      t = sh.red_u2[i];
      p = sh.red_p[i];
    }
  }
}

// Over the workgroup, in one exchange: whether any `flag` is set, the largest
// lo, the lowest token and its first position.
template <int kW>
__device__ __forceinline__ void block_bounds(Red<kW>& sh, uint32_t& flag, float& lo, uint32_t& t,
                                             uint32_t& p) {
  flag = __ballot(flag != 0u) != 0ull ? 1u : 0u;
  lo = wave_max(lo);
  wave_min_token(t, p);
  const int w = threadIdx.x / kWave;
  __syncthreads();
  if ((threadIdx.x % kWave) == 0) {
    sh.red_u[w] = flag;
    sh.red_f[w] = lo;
    sh.red_u2[w] = t;
    sh.red_p[w] = p;
  }
  __syncthreads();
  flag = sh.red_u[0];
  lo = sh.red_f[0];
  t = sh.red_u2[0];
  p = sh.red_p[0];
#pragma unroll
  for (int i = 1; i < kW; ++i) {
    flag |= sh.red_u[i];
    lo = __builtin_fmaxf(lo, sh.red_f[i]);
    if (sh.red_u2[i] < t) {
      t = sh.red_u2[i];
      p = sh.red_p[i];
    }
  }
}

__device__ __forceinline__ float half_lane(const uint4& q, int k) {
  const uint16_t* h = reinterpret_cast<const uint16_t*>(&q);
  return half_to_float(h[k]);
}

// Fast scores for H known at compile time: G lanes per candidate, each lane
// owning L = H / (8 G) 16-byte slices of the row (slice i*G + lane, so a group
// reads G*16 contiguous bytes per load), U candidates in flight per group.
// The lane's slice of y stays in registers for the whole block.
template <int H, int G, int U>
__device__ void fast_scores_vec(const HeadArgs& a, const float* ys,
                                HeadShared& sh, uint32_t n) {
  constexpr int L = H / (8 * G);
  constexpr int kGroups = kHeadThreads / G;
  static_assert(L * 8 * G == H, "H must split into 16-byte lane slices");
  const int lane = threadIdx.x % G;
  const int grp = threadIdx.x / G;
  float yv[L][8];
#pragma unroll
  for (int i = 0; i < L; ++i) {
#pragma unroll
    for (int k = 0; k < 8; ++k) yv[i][k] = ys[(i * G + lane) * 8 + k];
  }
  for (uint32_t base = 0; base < n; base += kGroups * U) {
    uint4 ev[U][L];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t c = base + u * kGroups + grp;
      ok[u] = c < n;
      const uint32_t t = ok[u] ? sh.tk[c] : 0u;
      const uint4* row = reinterpret_cast<const uint4*>(a.emb + static_cast<uint64_t>(t) * H) + lane;
#pragma unroll
      for (int i = 0; i < L; ++i) {
        ev[u][i] = ok[u] ? row[i * G] : uint4{0u, 0u, 0u, 0u};
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float acc = 0.0f;
      float acca = 0.0f;
#pragma unroll
      for (int i = 0; i < L; ++i) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float e = half_lane(ev[u][i], k);
          acc = __builtin_fmaf(e, yv[i][k], acc);
          acca = __builtin_fmaf(__builtin_fabsf(e), __builtin_fabsf(yv[i][k]), acca);
        }
      }
#pragma unroll
      for (int m = G / 2; m > 0; m >>= 1) {
        acc += __shfl_xor(acc, m, G);
        acca += __shfl_xor(acca, m, G);
      }
      const uint32_t c = base + u * kGroups + grp;
      if (lane == 0 && ok[u]) {
        sh.sc[c] = acc;
        sh.bd[c] = __builtin_fmaf(a.coef, acca, a.slack);
      }
    }
  }
}

// Fast scores for any H of whole 16-byte words: a wave takes U candidates at
// a time, each lane every 64th word of each row (contiguous reads, U loads in
// flight beside the hidden row's words from LDS).
template <int U>
__device__ void fast_scores_words(const HeadArgs& a, const float* ys, HeadShared& sh, uint32_t n) {
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t w = threadIdx.x / kWave;
  const uint32_t words = a.H / 8u;
  for (uint32_t base = w * U; base < n; base += kHeadWaves * U) {
    const uint4* row[U];
    float acc[U];
    float acca[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {  // past the end: the last candidate again
      const uint32_t c = base + u < n ? base + u : n - 1u;
      row[u] = reinterpret_cast<const uint4*>(a.emb + static_cast<uint64_t>(sh.tk[c]) * a.H);
      acc[u] = 0.0f;
      acca[u] = 0.0f;
    }
    for (uint32_t q = lane; q < words; q += kWave) {
      uint4 ev[U];
#pragma unroll
      for (int u = 0; u < U; ++u) ev[u] = row[u][q];
      const float4 y0 = reinterpret_cast<const float4*>(ys)[2u * q];
      const float4 y1 = reinterpret_cast<const float4*>(ys)[2u * q + 1u];
      const float yv[8] = {y0.x, y0.y, y0.z, y0.w, y1.x, y1.y, y1.z, y1.w};
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float e = half_lane(ev[u], k);
          acc[u] = __builtin_fmaf(e, yv[k], acc[u]);
          acca[u] = __builtin_fmaf(__builtin_fabsf(e), __builtin_fabsf(yv[k]), acca[u]);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float g = wave_sum_f32(acc[u]);
      const float m = wave_sum_f32(acca[u]);
      if (lane == 0 && base + u < n) {
        sh.sc[base + u] = g;
        sh.bd[base + u] = __builtin_fmaf(a.coef, m, a.slack);
      }
    }
  }
}

// Fast scores for any H: one wave per candidate, element-strided.
template <typename Y>
__device__ void fast_scores_generic(const HeadArgs& a, Y ys, HeadShared& sh, uint32_t n) {
  const int lane = threadIdx.x % kWave;
  const int w = threadIdx.x / kWave;
  for (uint32_t c = w; c < n; c += kHeadWaves) {
    const uint16_t* row = a.emb + static_cast<uint64_t>(sh.tk[c]) * a.H;
    float acc = 0.0f;
    float acca = 0.0f;
    for (uint32_t f = lane; f < a.H; f += kWave) {
      const float e = half_to_float(row[f]);
      acc = __builtin_fmaf(e, ys[f], acc);
      acca = __builtin_fmaf(__builtin_fabsf(e), __builtin_fabsf(ys[f]), acca);
    }
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) {
      acc += __shfl_xor(acc, m);
      acca += __shfl_xor(acca, m);
    }
    if (lane == 0) {
      sh.sc[c] = acc;
      sh.bd[c] = __builtin_fmaf(a.coef, acca, a.slack);
    }
  }
}

template <int kH, int kG, typename Y>
__device__ void fast_scores(const HeadArgs& a, Y ys, HeadShared& sh, uint32_t n) {
  if constexpr (kH > 0) {
    fast_scores_vec<kH, kG, 1>(a, ys, sh, n);
  } else if constexpr (kG == 8) {
    fast_scores_words<4>(a, ys, sh, n);
  } else {
    fast_scores_generic(a, ys, sh, n);
  }
}

// Summarises one block of n candidates (scores in sh.sc / sh.bd, ids in
// sh.tk, list positions pos0 + c) into sh.rec.  All threads must call.
template <typename Y>
__device__ void summarize_block(const HeadArgs& a, Y ys, HeadShared& sh, uint32_t n,
                                uint32_t pos0, bool invalid) {
  const int tid = threadIdx.x;
  if (invalid) {
    if (tid == 0) {
      sh.rec = Record{__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""),
                      kInvalidToken, 0u, kRecInvalid, kInvalidToken, 0u};
    }
    __syncthreads();
    return;
  }
  // pass 1: finiteness, best lower bound L, lowest id
  uint32_t finite = 1u;
  float lo = -__builtin_huge_valf();
  uint32_t mt = kInvalidToken;
  uint32_t mp = 0u;
  for (uint32_t c = tid; c < n; c += kHeadThreads) {
    const float g = sh.sc[c];
    const float b = sh.bd[c];
    const bool ok = __builtin_isfinite(g) && __builtin_isfinite(b) && b < 0x1p100f;
    finite &= ok ? 1u : 0u;
    lo = __builtin_fmaxf(lo, g - b);
    if (sh.tk[c] < mt) {
      mt = sh.tk[c];
      mp = pos0 + c;
    }
  }
  uint32_t bad = finite ^ 1u;
  block_bounds(sh, bad, lo, mt, mp);
  const bool all_finite = bad == 0u;
  const float L = lo;
  if (tid == 0) sh.n_members = 0u;
  __syncthreads();
  // pass 2: the window {g + b >= L}; everything when not all finite
  for (uint32_t c = tid; c < n; c += kHeadThreads) {
    const bool member = !all_finite || (sh.sc[c] + sh.bd[c] >= L);
    if (member) {
      const uint32_t slot = atomicAdd(&sh.n_members, 1u);
      sh.members[slot] = c;
    }
  }
  __syncthreads();
  const uint32_t nm = sh.n_members;
  if (all_finite && nm == 1u) {
    if (tid == 0) {
      const uint32_t c = sh.members[0];
      const float g = sh.sc[c];
      const float b = sh.bd[c];
      sh.rec = Record{g - b, g + b, g, sh.tk[c], pos0 + c, kRecFast, mt, mp};
    }
    __syncthreads();
    return;
  }
  // ambiguous window (or non-finite inputs): reference-order rescore
  Best best = best_identity();
  for (uint32_t i = tid; i < nm; i += kHeadThreads) {
    const uint32_t c = sh.members[i];
    const uint32_t t = sh.tk[c];
    const float s = canonical_dot_order(a.order, ys, a.emb + static_cast<uint64_t>(t) * a.H, a.H);
    best = best_of(best, best_leaf(s, t, pos0 + c));
  }
  best = block_best(sh, best);
  if (tid == 0) {
    if (best.token == kInvalidToken) {
      const float nan = __builtin_nanf("");
      sh.rec = Record{nan, nan, nan, kInvalidToken, 0u, kRecAllNan, mt, mp};
    } else {
      sh.rec = Record{best.score, best.score, best.score, best.token, best.pos,
                      kRecExact, mt, mp};
    }
  }
  __syncthreads();
}

// Merges n records of one row (in sh.recs) into one: invalid when any is;
// otherwise the exact best (reference-order score) of the records whose
// window reaches the best lower bound L (fast records rescored), or "all
// NaN" when none has a finite score; the lowest id of all of them rides
// along.  A fast record that is alone in the window stays as it is: its
// candidate is the winner, whatever its reference-order score.  Merging in stages gives the same record as merging all at once:
// L never exceeds the row's best exact score, so no stage drops the winner.
// All threads must call; every thread gets the record.
template <typename Y>
__device__ __forceinline__ Record merge_records(const HeadArgs& a, Y ys, HeadShared& sh, uint32_t n) {
  const int tid = threadIdx.x;
  uint32_t inv = 0u;
  float lo = -__builtin_huge_valf();
  uint32_t mt = kInvalidToken;
  uint32_t mp = 0u;
  for (uint32_t i = tid; i < n; i += kHeadThreads) {
    const Record& q = sh.recs[i];
    inv |= (q.kind & kRecInvalid) ? 1u : 0u;
    if (q.kind & (kRecFast | kRecExact)) lo = __builtin_fmaxf(lo, q.lower);
    if (q.min_token < mt) {
      mt = q.min_token;
      mp = q.min_pos;
    }
  }
  block_bounds(sh, inv, lo, mt, mp);
  const bool invalid = inv != 0u;
  const float L = lo;
  const float nan = __builtin_nanf("");
  if (invalid) return Record{nan, nan, nan, kInvalidToken, 0u, kRecInvalid, mt, mp};
  uint32_t in_window = 0u;
  for (uint32_t i = tid; i < n; i += kHeadThreads) {
    const Record& q = sh.recs[i];
    if ((q.kind & (kRecFast | kRecExact)) && q.upper >= L) {
      ++in_window;
      sh.rec = q;  // read back only if it is the only one
    }
  }
  if (block_sum(sh, in_window) == 1u) {
    Record m = sh.rec;
    m.min_token = mt;
    m.min_pos = mp;
    return m;
  }
  Best best = best_identity();
  for (uint32_t i = tid; i < n; i += kHeadThreads) {
    const Record& q = sh.recs[i];
    if ((q.kind & (kRecFast | kRecExact)) && q.upper >= L) {
      const float s = (q.kind & kRecExact)
                          ? q.value
                          : canonical_dot_order(a.order, ys,
                                                a.emb + static_cast<uint64_t>(q.token) * a.H, a.H);
      best = best_of(best, best_leaf(s, q.token, q.pos));
    }
  }
  best = block_best(sh, best);
  if (best.token == kInvalidToken) return Record{nan, nan, nan, kInvalidToken, 0u, kRecAllNan, mt, mp};
  return Record{best.score, best.score, best.score, best.token, best.pos, kRecExact, mt, mp};
}

// Merges the row's records (sh.recs[0, n)) and writes its outputs.
template <typename Y>
__device__ __forceinline__ void finalize_row(const HeadArgs& a, uint32_t r, Y ys, HeadShared& sh, uint32_t n) {
  const Record m = n == 1u ? sh.recs[0] : merge_records(a, ys, sh, n);
  if (threadIdx.x == 0) {
    uint32_t token = kInvalidToken;
    float score = __builtin_nanf("");
    if (m.kind & kRecExact) {
      token = m.token;
      score = m.value;
    } else if (m.kind & kRecFast) {
      // (the reference-order score, a chain of H steps, only where it is asked for)
      token = m.token;
      if (a.out_score != nullptr) {
        score = canonical_dot_order(a.order, ys, a.emb + static_cast<uint64_t>(m.token) * a.H, a.H);
      }
    } else if (m.kind & kRecAllNan) {
      // every score NaN: the lowest id (greedy.cu:205-207)
      token = m.min_token;
      if (a.out_score != nullptr) {
        score = canonical_dot_order(a.order, ys, a.emb + static_cast<uint64_t>(m.min_token) * a.H, a.H);
      }
    }
    a.out_token[r] = token;
    if (a.out_score != nullptr) a.out_score[r] = score;
  }
}

// Loads the ids of candidates [begin, begin + n) into sh.tk; returns whether
// any id is outside the vocabulary (the reference marks the row invalid).
// first_id: entry threadIdx.x of the list, already loaded.
__device__ bool load_block_ids(const HeadArgs& a, const RowList& rl, HeadShared& sh,
                               uint32_t begin, uint32_t n, uint32_t first_id) {
  uint32_t bad = 0u;
  for (uint32_t c = threadIdx.x; c < n; c += kHeadThreads) {
    const uint32_t t = begin + c == threadIdx.x ? first_id : rl.ids[begin + c];
    bad |= t >= a.V ? 1u : 0u;
    sh.tk[c] = t < a.V ? t : 0u;
  }
  return block_sum(sh, bad) != 0u;
}

// One workgroup per row.  Bound: latency (count and ids, candidate rows,
// three exchanges between the waves), and at wide rows the candidate rows'
// bytes.  A winner alone in its window needs no reference-order score (the
// operator returns tokens), which was a chain of H steps over single global
// loads by one thread.  256 rows of up to 128 candidates at H = 576: 13.7 -> 10.7
// us; 200 rows of up to 128 at H = 960 154 -> 18.7, 256 rows of up to 512 at
// H = 2048 1753 -> 117 (whole words instead of 2-byte loads).  The row's
// candidates come in blocks of a.chunk, each block summarized into a record in LDS, then merged (finalize_row); when
// the records fill their LDS array, they are merged into its first entry
// and the row goes on (lists of any length).  kGlobalHidden: the hidden row
// is read from global memory in place of an FP32 copy in LDS (rows too wide
// for LDS).
template <int kH, int kG, bool kGlobalHidden>
__global__ __launch_bounds__(kHeadThreads) void head_kernel(HeadArgs a) {
  extern __shared__ __align__(16) float ys_lds[];
  __shared__ HeadShared sh;
  const uint32_t r = blockIdx.x;
  // the list's first ids beside its count (entries of the row's fixed width)
  const uint32_t first_id =
      a.fixed_ids[static_cast<uint64_t>(r) * a.max_allowed +
                  (threadIdx.x < a.max_allowed ? threadIdx.x : a.max_allowed - 1u)];
  const RowList rl = resolve_row(a, r);
  if (rl.status == 1) {
    if (threadIdx.x == 0) {
      a.out_token[r] = kInvalidToken;
      if (a.out_score != nullptr) a.out_score[r] = __builtin_nanf("");
    }
    return;
  }
  auto body = [&](auto ys) {
    const uint32_t nblocks = (rl.count + a.chunk - 1) / a.chunk;
    uint32_t nrec = 0;
    for (uint32_t blk = 0; blk < nblocks; ++blk) {
      const uint32_t begin = blk * a.chunk;
      const uint32_t n = rl.count - begin < a.chunk ? rl.count - begin : a.chunk;
      const bool invalid = load_block_ids(a, rl, sh, begin, n, first_id);
      if (!invalid) fast_scores<kH, kG>(a, ys, sh, n);
      __syncthreads();
      summarize_block(a, ys, sh, n, begin, invalid);
      if (threadIdx.x == 0) sh.recs[nrec] = sh.rec;
      __syncthreads();
      ++nrec;
      if (nrec == kHeadMaxRecords && blk + 1 < nblocks) {
        const Record m = merge_records(a, ys, sh, nrec);
        __syncthreads();
        if (threadIdx.x == 0) sh.recs[0] = m;
        __syncthreads();
        nrec = 1;
      }
    }
    finalize_row(a, r, ys, sh, nrec);
  };
  if constexpr (kGlobalHidden) {
    body(HalfRow{a.hidden16 + static_cast<uint64_t>(r) * a.H});
  } else {
    const uint16_t* hidden = a.hidden16 + static_cast<uint64_t>(r) * a.H;
    if (a.H % 8u == 0u && (reinterpret_cast<uintptr_t>(a.hidden16) & 15u) == 0u) {
      for (uint32_t q = threadIdx.x; q < a.H / 8u; q += kHeadThreads) {
        const uint4 h = reinterpret_cast<const uint4*>(hidden)[q];
        float4* to = reinterpret_cast<float4*>(ys_lds) + 2u * q;
        to[0] = float4{half_lane(h, 0), half_lane(h, 1), half_lane(h, 2), half_lane(h, 3)};
        to[1] = float4{half_lane(h, 4), half_lane(h, 5), half_lane(h, 6), half_lane(h, 7)};
      }
    } else {
      for (uint32_t f = threadIdx.x; f < a.H; f += kHeadThreads) ys_lds[f] = half_to_float(hidden[f]);
    }
    __syncthreads();
    body(static_cast<const float*>(ys_lds));
  }
}

// ---------------------------------------------------------------------------
// Selection over precomputed logits (reference greedy.cu:21-131).
// ---------------------------------------------------------------------------

template <bool kHalf>
__device__ __forceinline__ float logit_at(const void* p, uint64_t i) {
  return kHalf ? half_to_float(static_cast<const uint16_t*>(p)[i])
               : static_cast<const float*>(p)[i];
}

// greedy_select: one workgroup of 1024 threads per row.  Bound: a row's bytes
// through one compute unit (there is no scratch memory to merge workgroups
// through: the reference's operator takes none), so what counts is the bytes
// in flight: kSelBatch 16-byte words per thread (128 KB per compute unit).
// Each thread keeps the first of its words that holds its best value (a word
// is compared by its maximum, NaN ignored), and only the threads whose best
// is the row's maximum look for the element.  A row may start anywhere: the
// elements before its first and after its last whole word are scalars.
// V = 49152 FP16: 8 rows 89.9 -> 4.4 us, 256 rows 89.0 -> 6.8 us (from one
// 2-byte load per thread and iteration in a 256-thread workgroup); one row of
// 128256: 6.8 us.
constexpr int kSelThreads = 1024;
constexpr uint32_t kSelBatch = 8;

// A signalling NaN would come out of a maximum as a NaN: made quiet first.
__device__ __forceinline__ half2_t quiet(uint32_t v) {
  return __builtin_elementwise_canonicalize(__builtin_bit_cast(half2_t, v));
}

// The largest value of a 16-byte word, NaN only if all are.
template <bool kHalf>
__device__ __forceinline__ float word_max(const uint4& q) {
  if constexpr (kHalf) {
    const half2_t m = __builtin_elementwise_max(
        __builtin_elementwise_max(quiet(q.x), quiet(q.y)),
        __builtin_elementwise_max(quiet(q.z), quiet(q.w)));
    return __builtin_fmaxf(static_cast<float>(m.x), static_cast<float>(m.y));
  } else {
    const float a = __builtin_fmaxf(__builtin_canonicalizef(as_float(q.x)),
                                    __builtin_canonicalizef(as_float(q.y)));
    const float b = __builtin_fmaxf(__builtin_canonicalizef(as_float(q.z)),
                                    __builtin_canonicalizef(as_float(q.w)));
    return __builtin_fmaxf(a, b);
  }
}

// Element k of a 16-byte word.
template <bool kHalf>
__device__ __forceinline__ float word_element(const uint4& q, uint32_t k) {
  const uint32_t w[4] = {q.x, q.y, q.z, q.w};
  if constexpr (kHalf) {
    return half_to_float(static_cast<uint16_t>(w[k / 2u] >> (16u * (k % 2u))));
  } else {
    return as_float(w[k]);
  }
}

template <bool kHalf>
__global__ __launch_bounds__(kSelThreads) void greedy_kernel(
    const void* __restrict__ logits, uint32_t* __restrict__ tokens, uint32_t V) {
  constexpr uint32_t kSize = kHalf ? 2u : 4u;
  constexpr uint32_t kPer = 16u / kSize;  // elements per word
  constexpr int kSelWaves = kSelThreads / kWave;
  __shared__ float red_f[kSelWaves];
  __shared__ uint32_t red_t[kSelWaves];
  const uint32_t tid = threadIdx.x;
  const uint64_t base = static_cast<uint64_t>(blockIdx.x) * V;
  const uintptr_t at = reinterpret_cast<uintptr_t>(logits) + base * kSize;
  // elements before the first whole word (all of them if no word is aligned)
  const uint32_t lead = static_cast<uint32_t>((0u - at) % 16u);
  const uint32_t head = (lead % kSize != 0u || lead / kSize > V) ? V : lead / kSize;
  const uint32_t words = (V - head) / kPer;
  const uint32_t tail = head + words * kPer;  // the first element after the words
  const uint4* row = reinterpret_cast<const uint4*>(at + static_cast<uintptr_t>(head) * kSize);

  const float low = -__builtin_huge_valf();
  float best = low;  // strictly greater wins: the first word of a thread's best value
  uint32_t word = 0u;
  uint4 hold{0u, 0u, 0u, 0u};
  for (uint32_t q0 = tid; q0 < words; q0 += kSelThreads * kSelBatch) {
    uint4 v[kSelBatch];
#pragma unroll
    for (uint32_t u = 0; u < kSelBatch; ++u) {  // past the end: the last word again
      const uint32_t q = q0 + u * kSelThreads;
      v[u] = row[q < words ? q : words - 1u];
    }
#pragma unroll
    for (uint32_t u = 0; u < kSelBatch; ++u) {
      const uint32_t q = q0 + u * kSelThreads;
      const float m = word_max<kHalf>(v[u]);
      if (m > best) {
        best = m;
        word = q < words ? q : words - 1u;
        hold = v[u];
      }
    }
  }
  float edge = low;  // the scalars of this thread, in ascending order
  uint32_t edge_token = kInvalidToken;
  for (uint64_t c = tid; c < head + (V - tail); c += kSelThreads) {
    const uint32_t t = static_cast<uint32_t>(c < head ? c : tail + (c - head));
    const float v = logit_at<kHalf>(logits, base + t);
    if (v > edge) {
      edge = v;
      edge_token = t;
    }
  }
  const float mine = wave_max(__builtin_fmaxf(best, edge));
  if (tid % kWave == 0u) red_f[tid / kWave] = mine;
  __syncthreads();
  float top = red_f[0];
#pragma unroll
  for (int i = 1; i < kSelWaves; ++i) top = __builtin_fmaxf(top, red_f[i]);
  uint32_t token = kInvalidToken;
  if (top > low) {
    if (edge == top) token = edge_token;
    if (best == top) {
#pragma unroll
      for (int k = static_cast<int>(kPer) - 1; k >= 0; --k) {
        const uint32_t t = head + word * kPer + static_cast<uint32_t>(k);
        if (word_element<kHalf>(hold, static_cast<uint32_t>(k)) == top && t < token) token = t;
      }
    }
  } else {  // nothing above -inf: the lowest -inf, or token 0 if all are NaN
    for (uint64_t c = tid; c < V && token == kInvalidToken; c += kSelThreads) {
      if (logit_at<kHalf>(logits, base + c) == low) token = static_cast<uint32_t>(c);
    }
  }
  token = wave_min_u32(token);
  if (tid % kWave == 0u) red_t[tid / kWave] = token;
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int i = 1; i < kSelWaves; ++i) token = __builtin_elementwise_min(token, red_t[i]);
    // src/cuda/greedy.cu:57: no comparable value selects token 0
    tokens[blockIdx.x] = token == kInvalidToken ? 0u : token;
  }
}

template <bool kHalf>
__global__ __launch_bounds__(kThreads) void restricted_greedy_kernel(
    const void* __restrict__ logits, const uint32_t* __restrict__ allowed,
    const uint32_t* __restrict__ counts, uint32_t* __restrict__ tokens,
    uint32_t V, uint32_t max_allowed) {
  __shared__ Red<kWaves> sh;
  const uint32_t r = blockIdx.x;
  const uint32_t count = counts[r];
  const bool row_invalid = count == 0 || count > max_allowed;
  const uint64_t base = static_cast<uint64_t>(r) * V;
  Best best = best_identity();
  uint32_t bad = 0u;
  uint32_t mt = kInvalidToken;
  uint32_t mp = 0u;
  if (!row_invalid) {
    for (uint32_t j = threadIdx.x; j < count; j += kThreads) {
      const uint32_t t = allowed[static_cast<uint64_t>(r) * max_allowed + j];
      if (t >= V) {
        bad = 1u;
        continue;
      }
      if (t < mt) {
        mt = t;
        mp = j;
      }
      best = best_of(best, best_leaf(logit_at<kHalf>(logits, base + t), t, j));
    }
  }
  const bool invalid = block_sum(sh, bad) != 0u || row_invalid;
  best = block_best(sh, best);
  block_min_token(sh, mt, mp);
  if (threadIdx.x == 0) {
    tokens[r] = invalid ? kInvalidToken : (best.token == kInvalidToken ? mt : best.token);
  }
}

__global__ __launch_bounds__(kThreads) void fill_zero_kernel(uint4* p, uint64_t n16) {
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x; i < n16;
       i += static_cast<uint64_t>(gridDim.x) * kThreads) {
    p[i] = uint4{0u, 0u, 0u, 0u};
  }
}

// Read floor: every 16 bytes of [p, p + 16 n16) read once, kReadBatch
// loads per thread issued before any is used, each workgroup on one
// contiguous chunk; the XOR of the words goes to *sink only if it equals a
// value that never occurs in practice (the loads must not be optimized away).
constexpr uint32_t kReadBatch = 8;
__global__ __launch_bounds__(kThreads) void read_floor_kernel(const uint4* p, uint64_t n16,
                                                              uint32_t* sink) {
  const uint64_t base = static_cast<uint64_t>(blockIdx.x) * kReadBatch * kThreads + threadIdx.x;
  uint4 v[kReadBatch];
#pragma unroll
  for (uint32_t u = 0; u < kReadBatch; ++u) {
    const uint64_t q = base + u * kThreads;
    v[u] = q < n16 ? p[q] : uint4{0u, 0u, 0u, 0u};
  }
  uint32_t x = 0u;
#pragma unroll
  for (uint32_t u = 0; u < kReadBatch; ++u) x ^= v[u].x ^ v[u].y ^ v[u].z ^ v[u].w;
  if (x == 0x9E3779B9u && threadIdx.x == 0) *sink = x;
}

} // namespace

hipError_t launch_read_floor(const void* address, uint64_t bytes, uint32_t* sink,
                             hipStream_t stream) {
  const uint64_t n16 = bytes / 16;
  if (n16 == 0) return hipSuccess;
  const uint64_t blocks = (n16 + kReadBatch * kThreads - 1) / (kReadBatch * kThreads);
  if (blocks > 0xFFFFFFFFull) return hipErrorInvalidValue;
  hipLaunchKernelGGL(read_floor_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kThreads), 0,
                     stream, static_cast<const uint4*>(address), n16, sink);
  return hipGetLastError();
}

// The split of rms_norm_rows_kernel, if the call is one for it: whole
// aligned 16-byte words per row, at most 64 segments of kNormSegMax words.
// As few lanes per row as hold it (fewer hand-overs, more rows per wave).
static bool norm_split(const void* input, const void* weight, const void* output, bool half,
                       uint32_t rows, uint32_t hidden, NormSplit& d, uint32_t& seg) {
  const uint32_t per = half ? 8u : 4u;
  if (hidden % per != 0 || hidden / per > kNormSegMax * kWave ||
      ((reinterpret_cast<uintptr_t>(input) | reinterpret_cast<uintptr_t>(weight) |
        reinterpret_cast<uintptr_t>(output)) & 15u) != 0) {
    return false;
  }
  d.words = hidden / per;
  d.lanes_log2 = 0;
  while (d.words > kNormSegMax << d.lanes_log2) ++d.lanes_log2;
  seg = (((d.words + (1u << d.lanes_log2) - 1u) >> d.lanes_log2) + 3u) & ~3u;
  d.per_wave = 1;
  while (rows / (2u * d.per_wave) >= kNormWaves && 2u * d.per_wave <= 64u >> d.lanes_log2) {
    d.per_wave *= 2u;
  }
  d.row_magic = ((1u << 20) + d.words - 1u) / d.words;
  return true;
}

template <bool kHalf>
static void launch_norm_rows(const void* input, const void* weight, void* output, uint32_t rows,
                             uint32_t hidden, float epsilon, const NormSplit& d, uint32_t seg,
                             hipStream_t stream) {
  const dim3 grid((rows + d.per_wave - 1u) / d.per_wave), block(kWave);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, stream, input, weight, output, rows, hidden, epsilon, d);
  };
  if (seg == 4u) {
    go(rms_norm_rows_kernel<kHalf, 4>);
  } else if (seg == 8u) {
    go(rms_norm_rows_kernel<kHalf, 8>);
  } else if (seg == 12u) {
    go(rms_norm_rows_kernel<kHalf, 12>);
  } else {
    go(rms_norm_rows_kernel<kHalf, 16>);
  }
}

hipError_t launch_rms_norm(const void* input, bool half_input, const void* weight,
                           bool half_weight, void* output, bool half_output,
                           float* row_norm, uint32_t rows, uint32_t hidden,
                           float epsilon, hipStream_t stream) {
  const dim3 grid(rows), block(kWave);
  NormSplit split{};
  uint32_t seg = 0;
  if (half_input == half_weight && half_input == half_output && row_norm == nullptr &&
      norm_split(input, weight, output, half_input, rows, hidden, split, seg)) {
    if (half_input) {
      launch_norm_rows<true>(input, weight, output, rows, hidden, epsilon, split, seg, stream);
    } else {
      launch_norm_rows<false>(input, weight, output, rows, hidden, epsilon, split, seg, stream);
    }
    return hipGetLastError();
  }
  if (hidden > kNormStagedMax) {
    if (row_norm != nullptr && hidden > 65536u) return hipErrorInvalidValue;  // bound's margin
    if (half_input && half_weight && half_output) {
      hipLaunchKernelGGL((rms_norm_wide_kernel<true, true, true>), grid, block, 0, stream,
                         input, weight, output, nullptr, hidden, epsilon);
    } else if (!half_input && !half_weight && !half_output) {
      hipLaunchKernelGGL((rms_norm_wide_kernel<false, false, false>), grid, block, 0, stream,
                         input, weight, output, row_norm, hidden, epsilon);
    } else {
      return hipErrorInvalidValue;
    }
    return hipGetLastError();
  }
  const size_t lds = (hidden <= kNormStagedWeightMax ? 3u : 2u) * static_cast<size_t>(hidden) *
                     sizeof(float);
  if (half_input && half_weight && half_output) {
    hipLaunchKernelGGL((rms_norm_kernel<true, true, true>), grid, block, lds, stream,
                       input, weight, output, nullptr, hidden, epsilon);
  } else if (!half_input && !half_weight && !half_output) {
    hipLaunchKernelGGL((rms_norm_kernel<false, false, false>), grid, block, lds, stream,
                       input, weight, output, row_norm, hidden, epsilon);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_head(const HeadArgs& args, hipStream_t stream) {
  const bool aligned = (reinterpret_cast<uintptr_t>(args.emb) & 15u) == 0;
  const size_t lds = static_cast<size_t>(args.H) * sizeof(float);
  if (args.H == 576 && aligned) {
    hipLaunchKernelGGL((head_kernel<576, 8, false>), dim3(args.rows), dim3(kHeadThreads), lds, stream, args);
  } else if (args.H % 8u == 0 && aligned && args.H <= kHeadLdsHidden) {
    hipLaunchKernelGGL((head_kernel<0, 8, false>), dim3(args.rows), dim3(kHeadThreads), lds, stream, args);
  } else if (args.H <= kHeadLdsHidden) {
    hipLaunchKernelGGL((head_kernel<0, 64, false>), dim3(args.rows), dim3(kHeadThreads), lds, stream, args);
  } else {
    hipLaunchKernelGGL((head_kernel<0, 64, true>), dim3(args.rows), dim3(kHeadThreads), 0, stream, args);
  }
  return hipGetLastError();
}

hipError_t launch_linear_f16_simple(const uint16_t* input, const uint16_t* weight,
                                    uint16_t* output, uint32_t rows, uint32_t in_features,
                                    uint32_t out_features, hipStream_t stream) {
  const uint64_t n = static_cast<uint64_t>(rows) * out_features;
  const uint64_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(linear_f16_simple_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0,
                     stream, input, weight, output, rows, in_features, out_features);
  return hipGetLastError();
}

hipError_t launch_greedy(const void* logits, bool half, uint32_t* tokens,
                         uint32_t rows, uint32_t vocab, hipStream_t stream) {
  if (half) {
    hipLaunchKernelGGL((greedy_kernel<true>), dim3(rows), dim3(kSelThreads), 0, stream,
                       logits, tokens, vocab);
  } else {
    hipLaunchKernelGGL((greedy_kernel<false>), dim3(rows), dim3(kSelThreads), 0, stream,
                       logits, tokens, vocab);
  }
  return hipGetLastError();
}

hipError_t launch_restricted_greedy(const void* logits, bool half,
                                    const uint32_t* allowed, const uint32_t* counts,
                                    uint32_t* tokens, uint32_t rows, uint32_t vocab,
                                    uint32_t max_allowed, hipStream_t stream) {
  if (half) {
    hipLaunchKernelGGL((restricted_greedy_kernel<true>), dim3(rows), dim3(kThreads), 0,
                       stream, logits, allowed, counts, tokens, vocab, max_allowed);
  } else {
    hipLaunchKernelGGL((restricted_greedy_kernel<false>), dim3(rows), dim3(kThreads), 0,
                       stream, logits, allowed, counts, tokens, vocab, max_allowed);
  }
  return hipGetLastError();
}

hipError_t launch_fill_zero(void* address, uint64_t bytes, hipStream_t stream) {
  const uint64_t n16 = bytes / 16;
  if (n16 == 0) return hipSuccess;
  uint64_t blocks = (n16 + kThreads - 1) / kThreads;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(fill_zero_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kThreads), 0,
                     stream, static_cast<uint4*>(address), n16);
  return hipGetLastError();
}

} // namespace mf
