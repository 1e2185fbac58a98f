// The full output projection on gfx950 MFMA: C[m, V] = A[m, H] . E[V, H]^T
// with FP16 A and E, FP32 accumulation, FP32 or FP16 (round to nearest
// even) output -- linear_f16 (the reference's cublasGemmEx call,
// src/cuda/linear.cu:92-102) of more than kStreamRowsMax rows and the
// full-vocabulary comparator's scores.
//
// Tiling.  A workgroup owns tiles of 256 A rows x kNT tokens (64, 128 or 192,
// launch_projection).  Eight MFMA waves, two a SIMD, each multiply 64 rows x
// kNT / 2 tokens as 4 x kNT / 32 blocks of v_mfma_f32_16x16x32_f16, so one
// wave's MFMAs run under the other's LDS reads.  The tokens are the first
// operand: a lane then holds four consecutive tokens of one row, or, for FP16
// results, with the token rows of a block pair interleaved (token_row), eight,
// which it stores as 16 bytes straight from its registers.
//
// K runs in chunks of 64 features (whole 128-byte lines).  A chunk's A rows
// and E rows go straight from memory into LDS by global_load_lds copies.  Four
// copy waves of their own issue them: vector memory operations end in order,
// so a wave that also stores results would wait for those before it could
// hand over the next chunk, and the stores of a tile (8 us of the chip's
// writes) would stop the multiplication.  LDS holds two and a half chunks of A
// rows (units of 128 rows through a ring of five, so that half of a chunk is
// on its way before its turn) and three of E rows, 152 KB at kNT = 192.  The
// 16-byte pieces of a row are XOR-swizzled so that the 16 lanes one
// ds_read_b128 cycle serves meet 16 bank groups (SQ_LDS_BANK_CONFLICT = 0).
// One barrier per chunk, where every wave has its last fragments in registers.
//
// The workgroups stay (one per compute unit) and run their tiles as one
// stream of chunks: the copies run on into the next tile while the last
// chunk is multiplied and the results stored.  The compute units of an XCD
// (blockIdx % 8) take the M-tiles of the same tokens side by side, so the E
// rows come from HBM once.
//
// Bound: the copies, 57 KB/us per compute unit alone (copies only, 1.1 us a
// chunk of 64 KB) against 0.7 us of MFMAs; with both, 1.4 us.  Measured (FP16
// output, calls, from 32-feature chunks and 32x32x16 MFMAs in four waves):
// 1024 x 2048 x 128256 688 -> 482-497 us (1.10 PFLOP/s; hipBLASLt 530),
// 512 x 1024 x 120000 163 -> 133, 256 x 2048 x 50021 118 -> 83,
// 256 x 576 x 49152 20.6 -> 19.9.  Tried: the copies in the MFMA waves (544 us at
// kNT = 256; with the fragments a half chunk ahead 570, with the ring of five
// 567), priorities for four of the MFMA waves or for the copy waves (512, 519
// against 511).
//
// The comparator also needs ||e_t|| per token for its error bound: the waves
// of the first rows of M-tile 0 sum the squares of the E fragments they read
// (FP32, any order; the (1 + 2^-7) factor of the bound covers it).
#include <hip/hip_runtime.h>

#include "mf_device.hpp"
#include "mf_launch.hpp"

namespace mf {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kMmaWaves = 8;
constexpr uint32_t kCopyWaves = 4;
constexpr int kThreads = static_cast<int>(64u * (kMmaWaves + kCopyWaves));
constexpr uint32_t kMT = 256;            // A rows per tile
constexpr uint32_t kWaveRows = 64;       // and per wave: wave w takes rows 64 (w % 4) ..
constexpr uint32_t kRB = kWaveRows / 16u;
constexpr uint32_t kKC = 64;             // features per chunk
constexpr uint32_t kRow = kKC * 2u;      // bytes of a row in a chunk
// An operand's rows per chunk, copied in kUnits units through a ring.
template <uint32_t kRows>
struct Ring {
  static constexpr uint32_t kUnits = kRows == 256u ? 2u : 1u;
  static constexpr uint32_t kSlots = 2u * kUnits + 1u;
  static constexpr uint32_t kUnitRows = kRows / kUnits;
  static constexpr uint32_t kBytes = kUnitRows * kRow;
  static constexpr uint32_t kCopies = kBytes / 1024u / kCopyWaves;  // 1 KiB copies per wave and unit
  static_assert(kBytes % (1024u * kCopyWaves) == 0, "every wave issues the same copies");
};

template <uint32_t kNT>
constexpr uint32_t kGemmLds = Ring<kMT>::kSlots * Ring<kMT>::kBytes + Ring<kNT>::kSlots * Ring<kNT>::kBytes;
static_assert(kGemmLds<192> <= 160u * 1024u, "LDS");

// The piece p of A row r sits at p ^ a_swz(r), of E row t at p ^ b_swz(t).
// A fragment reads 16 consecutive A rows, or, where the result is FP16 (kPair),
// E rows 8 i + {0..3} (+ 4), else 16 consecutive ones as well.
__device__ __forceinline__ uint32_t a_swz(uint32_t r) { return (r >> 1) & 7u; }
template <bool kPair>
__device__ __forceinline__ uint32_t b_swz(uint32_t t) {
  return kPair ? ((t >> 1) & 1u) | ((t >> 2) & 6u) : (t >> 1) & 7u;
}
// Token (of 32) that row i of block 0 or 1 of a pair holds.  A lane's results
// are 16 bytes of consecutive tokens either way: eight FP16 of a block pair,
// or four FP32 of each block.  One store instruction then fills whole 64-byte
// pieces of a row.  With pairs for FP32 too, every store left half of each
// 32 bytes to the next one: the product of 256 x 576 x 49152, written through,
// took 59 us, and the comparator's step around it 86 instead of 53.
template <bool kPair>
__device__ __forceinline__ uint32_t token_row(uint32_t block, uint32_t i) {
  return kPair ? 8u * (i / 4u) + 4u * block + i % 4u : 16u * block + i;
}

// Wait until at most kN of this wave's vector memory operations are in flight.
template <int kN>
__device__ __forceinline__ void wait_copies() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kN) : "memory");
}

// A workgroup barrier without __syncthreads' release fence, which would wait
// for every copy in flight.  The wave's own LDS operations are complete when
// it arrives.
__device__ __forceinline__ void chunk_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// FP16 results of tiles of few chunks are written through to memory (whole rows
// of 16-byte words only): the workgroups' stores then come close together, and
// what stays dirty in L2 is written back after the last of them.  FP32 scores
// are read by the selection that follows (comparator of 256 rows at H = 576,
// V = 49152: 53.3 us, written through 54.6).
constexpr uint32_t kThroughChunks = 15;

// 16 bytes to global memory at any element (gfx950 stores need no alignment).
struct __attribute__((packed, aligned(2))) Any16 {
  u32x4 v;
};
template <bool kThrough>
__device__ __forceinline__ void store16(void* dst, u32x4 v) {
  if constexpr (kThrough) {
    // (the store reads its registers late: two wait states before a vector
    // instruction may write them, which the compiler does not see here)
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1 nt\n\ts_nop 1" ::"v"(dst), "v"(v) : "memory");
  } else {
    static_cast<Any16*>(dst)->v = v;
  }
}

template <uint32_t kNT, bool kF16Out>
__global__ __launch_bounds__(kThreads) void projection_kernel(ProjArgs a, uint32_t n_tiles,
                                                                 uint32_t m_tiles) {
  using RA = Ring<kMT>;
  using RB = Ring<kNT>;
  constexpr uint32_t kWaveTokens = kNT / 2u;
  constexpr uint32_t kTB = kWaveTokens / 16u;
  extern __shared__ __align__(16) unsigned char lds[];
  unsigned char* const abase = lds;
  unsigned char* const bbase = lds + RA::kSlots * RA::kBytes;
  const uint32_t lane = threadIdx.x % 64u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64u);
  const uint32_t wm = wave % 4u;  // rows 64 wm .. of the tile
  const uint32_t wn = wave / 4u;  // tokens kWaveTokens wn ..
  const uint32_t col = lane % 16u;
  const uint32_t kb = lane / 16u;
  const uint32_t chunks = (a.H + kKC - 1u) / kKC;

  // this workgroup's tiles: XCD x takes the token tiles n = x (mod 8), its
  // compute units tile j = idx, idx + per_xcd, .. of them, M-tile fastest
  const uint32_t x = blockIdx.x % 8u;
  const uint32_t idx = blockIdx.x / 8u;
  const uint32_t per_xcd = gridDim.x / 8u;
  const uint32_t x_tiles = (n_tiles > x ? (n_tiles - x + 7u) / 8u : 0u) * m_tiles;
  if (idx >= x_tiles) return;
  const uint32_t total = ((x_tiles - idx + per_xcd - 1u) / per_xcd) * chunks;

  if (wave >= kMmaWaves) {
    // copy i of this wave in a unit: rows 8 (cw + 4 i) ..; lane l brings row
    // l / 8 of them, LDS piece l % 8
    const uint32_t cw = wave - kMmaWaves;
    const uint32_t cr = 8u * cw + lane / 8u;
    struct Stream {  // the next unit of an operand to copy
      uint32_t j, c, unit, slot;
    };
    Stream sa{idx, 0u, 0u, 0u}, sb{idx, 0u, 0u, 0u};
    auto advance = [&](Stream& s, uint32_t units, uint32_t slots) {
      if (++s.unit == units) {
        s.unit = 0u;
        if (++s.c == chunks) {
          s.c = 0u;
          s.j += per_xcd;
        }
      }
      if (++s.slot == slots) s.slot = 0u;
    };
    // past the row's end (a last half chunk) a piece re-reads the half before
    auto feature = [&](uint32_t c, uint32_t p) {
      const uint32_t k = c * kKC + p * 8u;
      return k < a.H ? k : k - 32u;
    };
    auto issue_a = [&]() {
      const uint32_t m0 = (sa.j % m_tiles) * kMT + sa.unit * RA::kUnitRows;
      unsigned char* buf = abase + sa.slot * RA::kBytes;
#pragma unroll
      for (uint32_t i = 0; i < RA::kCopies; ++i) {
        const uint32_t r = cr + 8u * kCopyWaves * i;
        const uint32_t row = m0 + r < a.m ? m0 + r : a.m - 1u;
        burst_to_lds(a.a16 + static_cast<uint64_t>(row) * a.H + feature(sa.c, (lane % 8u) ^ a_swz(r)),
                     buf + (cw + kCopyWaves * i) * 1024u);
      }
      advance(sa, RA::kUnits, RA::kSlots);
    };
    auto issue_b = [&]() {
      const uint32_t n0 = ((sb.j / m_tiles) * 8u + x) * kNT + sb.unit * RB::kUnitRows;
      unsigned char* buf = bbase + sb.slot * RB::kBytes;
#pragma unroll
      for (uint32_t i = 0; i < RB::kCopies; ++i) {
        const uint32_t t = cr + 8u * kCopyWaves * i;
        const uint32_t tok = n0 + t < a.V ? n0 + t : a.V - 1u;
        burst_to_lds(a.emb + static_cast<uint64_t>(tok) * a.H + feature(sb.c, (lane % 8u) ^ b_swz<kF16Out>(t)),
                     buf + (cw + kCopyWaves * i) * 1024u);
      }
      advance(sb, RB::kUnits, RB::kSlots);
    };
    // the part of a chunk that was not copied ahead of the one before it, then
    // the part of the next chunk that is
    auto issue_rest = [&]() {
      issue_a();
    };
    auto issue_ahead = [&]() {
      issue_a();
      issue_b();
    };
    constexpr int kAhead = static_cast<int>(RA::kCopies + RB::kCopies);
    constexpr int kRest = static_cast<int>(RA::kCopies);

    // chunks 0, 1 and the part of chunk 2 that fits
    issue_ahead();
    issue_rest();
    if (total > 1u) {
      issue_ahead();
      issue_rest();
      if (total > 2u) {
        issue_ahead();
        wait_copies<2 * kAhead + kRest>();
      } else {
        wait_copies<kAhead + kRest>();
      }
    } else {
      wait_copies<0>();
    }
    chunk_barrier();  // chunk 0 in LDS
    for (uint32_t q = 0; q < total; ++q) {
      // chunk q + 1 has landed (in flight: what was copied ahead of q + 2)
      if (q + 2u < total) {
        wait_copies<kAhead>();
      } else {
        wait_copies<0>();
      }
      chunk_barrier();  // chunk q read by every MFMA wave
      if (q + 2u < total) issue_rest();  // into chunk q's slots
      if (q + 3u < total) issue_ahead();
    }
    return;
  }

  floatx4 acc[kTB][kRB];
  float tok_sq[kTB];
  auto clear = [&]() {
#pragma unroll
    for (uint32_t i = 0; i < kTB; ++i) {
      tok_sq[i] = 0.0f;
#pragma unroll
      for (uint32_t j = 0; j < kRB; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  };
  clear();

  // a chunk's fragments come in two halves of 32 features
  struct Half {
    half8_t a[kRB];
    half8_t b[kTB];
  };
  uint32_t as = 0, bs = 0;  // the slots of the chunk's first units
  // this wave's rows and tokens: their units, and places in them
  const uint32_t au = kWaveRows * wm / RA::kUnitRows;
  const uint32_t bu = kWaveTokens * wn / RB::kUnitRows;
  const uint32_t ar = kWaveRows * wm % RA::kUnitRows + col;
  const uint32_t br = kWaveTokens * wn % RB::kUnitRows;
  auto read_half = [&](uint32_t h, Half& f) {
    const uint32_t aslot = as + au < RA::kSlots ? as + au : as + au - RA::kSlots;
    const uint32_t bslot = bs + bu < RB::kSlots ? bs + bu : bs + bu - RB::kSlots;
    const unsigned char* abuf = abase + aslot * RA::kBytes;
    const unsigned char* bbuf = bbase + bslot * RB::kBytes;
    const uint32_t p = 4u * h + kb;
#pragma unroll
    for (uint32_t j = 0; j < kRB; ++j) {
      const uint32_t r = ar + 16u * j;
      f.a[j] = *reinterpret_cast<const half8_t*>(abuf + r * kRow + (p ^ a_swz(r)) * 16u);
    }
#pragma unroll
    for (uint32_t i = 0; i < kTB; ++i) {
      const uint32_t t = br + 32u * (i / 2u) + token_row<kF16Out>(i % 2u, col);
      f.b[i] = *reinterpret_cast<const half8_t*>(bbuf + t * kRow + (p ^ b_swz<kF16Out>(t)) * 16u);
    }
  };
  bool norms = false;
  auto multiply = [&](const Half& f) {
#pragma unroll
    for (uint32_t i = 0; i < kTB; ++i) {
#pragma unroll
      for (uint32_t j = 0; j < kRB; ++j) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.b[i], f.a[j], acc[i][j], 0, 0, 0);
      }
    }
    if constexpr (!kF16Out) {
      if (norms) {
#pragma unroll
        for (uint32_t i = 0; i < kTB; ++i) {
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const float e = static_cast<float>(f.b[i][k]);
            tok_sq[i] = __builtin_fmaf(e, e, tok_sq[i]);
          }
        }
      }
    }
  };

  chunk_barrier();
  const bool through = kF16Out && chunks <= kThroughChunks && a.V % 8u == 0u;
  uint32_t c = 0, j_tile = idx;
  for (uint32_t q = 0; q < total; ++q) {
    norms = !kF16Out && a.tok_norm != nullptr && wm == 0u && j_tile % m_tiles == 0u;
    Half f;
    read_half(0u, f);
    multiply(f);
    read_half(1u, f);
    chunk_barrier();  // every read of chunk q has arrived; chunk q + 1 in LDS
    if ((as += RA::kUnits) >= RA::kSlots) as -= RA::kSlots;
    if ((bs += RB::kUnits) >= RB::kSlots) bs -= RB::kSlots;
    if (c * kKC + 32u < a.H) multiply(f);
    if (++c < chunks) continue;
    c = 0u;
    // the tile's results: block i, row block j: lane l holds tokens
    // token_row(i % 2, 4 (l / 16) + e), e = 0..3, of row 16 j + l % 16
    const uint32_t m0 = (j_tile % m_tiles) * kMT + kWaveRows * wm;
    const uint32_t n0 = ((j_tile / m_tiles) * 8u + x) * kNT + kWaveTokens * wn;
    uint32_t el = lane;  // (opaque: its parts are formed here, not held over the chunks)
    asm volatile("" : "+v"(el));
    const uint32_t ecol = el % 16u;
    const uint32_t ekb = el / 16u;
    if constexpr (!kF16Out) {
      if (norms) {
#pragma unroll
        for (uint32_t i = 0; i < kTB; ++i) {  // the K quarters of a token: lanes l, l ^ 16, l ^ 32
          float sq = tok_sq[i];
          sq += __shfl_xor(sq, 16);
          sq += __shfl_xor(sq, 32);
          const uint32_t tok = n0 + 32u * (i / 2u) + token_row<kF16Out>(i % 2u, ecol);
          if (ekb == 0u && tok < a.V) a.tok_norm[tok] = __fsqrt_rn(sq) * (1.0f + 0x1p-7f);
        }
      }
    }
    constexpr uint32_t kLaneBlocks = kF16Out ? 2u : 1u;
    constexpr uint32_t kLaneTokens = 4u * kLaneBlocks;
    auto store = [&]<bool kThrough>() {
#pragma unroll
      for (uint32_t j = 0; j < kRB; ++j) {
        const uint32_t row = m0 + 16u * j + ecol;
        const uint64_t at = static_cast<uint64_t>(row) * a.V;
#pragma unroll
        for (uint32_t i = 0; i < kTB; i += kLaneBlocks) {
          const uint32_t tok = n0 + 16u * i + kLaneTokens * ekb;  // this lane's tokens
          if (row >= a.m || tok >= a.V) continue;
          if (a.V - tok >= kLaneTokens) {  // (16-byte stores at any element: rows of odd V too)
            if constexpr (kF16Out) {
              u32x4 v;
#pragma unroll
              for (uint32_t e = 0; e < 4u; ++e) {
                const floatx4& s = e < 2u ? acc[i][j] : acc[i + 1u][j];
                v[e] = static_cast<uint32_t>(float_to_half_rne(s[2u * (e % 2u)])) |
                       (static_cast<uint32_t>(float_to_half_rne(s[2u * (e % 2u) + 1u])) << 16);
              }
              store16<kThrough>(a.out_f16 + at + tok, v);
            } else {
              store16<kThrough>(a.out_f32 + at + tok, __builtin_bit_cast(u32x4, acc[i][j]));
            }
          } else {
#pragma unroll
            for (uint32_t e = 0; e < kLaneTokens; ++e) {
              const float s = acc[i + e / 4u][j][e % 4u];
              if (tok + e < a.V) {
                if constexpr (kF16Out) {
                  a.out_f16[at + tok + e] = float_to_half_rne(s);
                } else {
                  a.out_f32[at + tok + e] = s;
                }
              }
            }
          }
        }
      }
    };
    if (through) {
      store.template operator()<true>();
    } else {
      store.template operator()<false>();
    }
    clear();
    j_tile += per_xcd;
  }
}

// Time of the whole grid with kNT-token tiles, in rows copied per compute
// unit: the rounds of the persistent workgroups, each a tile's A and E rows.
uint64_t grid_rows(const ProjArgs& a, uint32_t nt, uint32_t m_tiles, uint32_t per_xcd) {
  const uint64_t n_tiles = (static_cast<uint64_t>(a.V) + nt - 1u) / nt;
  const uint64_t rounds = ((n_tiles + 7u) / 8u * m_tiles + per_xcd - 1u) / per_xcd;
  return rounds * (kMT + nt);
}

template <uint32_t kNT>
hipError_t launch_tiles(const ProjArgs& a, uint32_t m_tiles, uint32_t per_xcd, hipStream_t stream) {
  const uint32_t n_tiles = (a.V + kNT - 1u) / kNT;
  const dim3 grid(per_xcd * 8u);
  if (a.out_f16 != nullptr) {
    hipLaunchKernelGGL((projection_kernel<kNT, true>), grid, dim3(kThreads), kGemmLds<kNT>, stream, a,
                       n_tiles, m_tiles);
  } else {
    hipLaunchKernelGGL((projection_kernel<kNT, false>), grid, dim3(kThreads), kGemmLds<kNT>, stream, a,
                       n_tiles, m_tiles);
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_projection(const ProjArgs& args, uint32_t groups, hipStream_t stream) {
  if (args.H % 32u != 0 || args.H == 0 || args.m == 0 || args.V == 0 || args.a16 == nullptr ||
      args.emb == nullptr || (args.out_f32 == nullptr) == (args.out_f16 == nullptr) || groups < 8u ||
      reinterpret_cast<uintptr_t>(args.a16) % 16u != 0 ||
      reinterpret_cast<uintptr_t>(args.emb) % 16u != 0) {
    return hipErrorInvalidValue;
  }
  const uint32_t per_xcd = groups / 8u;
  const uint32_t m_tiles = (args.m + kMT - 1u) / kMT;
  const uint64_t r192 = grid_rows(args, 192, m_tiles, per_xcd);
  const uint64_t r128 = grid_rows(args, 128, m_tiles, per_xcd);
  const uint64_t r64 = grid_rows(args, 64, m_tiles, per_xcd);
  // (a workgroup's chunks are counted in 32 bits)
  if (r64 / kMT * ((args.H + kKC - 1u) / kKC) > 0xFFFFFFFFull) return hipErrorInvalidValue;
  if (r192 <= r128 && r192 <= r64) return launch_tiles<192>(args, m_tiles, per_xcd, stream);
  if (r128 <= r64) return launch_tiles<128>(args, m_tiles, per_xcd, stream);
  return launch_tiles<64>(args, m_tiles, per_xcd, stream);
}

}  // namespace mf
