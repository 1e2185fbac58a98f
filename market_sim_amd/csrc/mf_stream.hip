// Few rows against the whole table on gfx950 MFMA: the table streams once
// through LDS past at most 128 A rows.  Two uses:
//   * the head of the unrestricted rows (stream_kernel<64, true>): the FP16
//     hi and lo of 32 slots as A rows, reduced in a windowed-argmax epilogue
//     to one window record per (slot, tile);
//   * linear_f16 of few rows (stream_kernel<kMT, false>), FP16 output.
//
// Bound: HBM for the table.  What that asks for is that every compute unit
// streams all the time and that all end together:
//   * tiles of 16 nb tokens, nb chosen so that the vocabulary's tiles fill
//     whole rounds of 256 compute units (stream_tile_blocks): a fixed tile of
//     192 tokens left V = 50021 with 261 tiles, 2 rounds for 5 of them;
//   * four copy waves bring a tile's rows into a ring of LDS chunks (64
//     features: whole 128-byte lines) with global_load_lds and run on across
//     tile boundaries, nbuf - 1 chunks ahead, so the epilogue of a tile does
//     not stop the stream; four MFMA waves read the chunks;
//   * one barrier per chunk (an s_barrier without __syncthreads' release
//     fence, which would wait for every copy in flight).
// A chunk's rows (A rows, then tokens) are 128 bytes each, the 16-byte pieces
// XOR-swizzled by the row's bits 1-3: the 16 lanes one ds_read_b128 cycle
// serves then meet 16 different bank groups.
//
// Measured (calls, tables partly in the last-level cache): linear_f16 of 1, 32,
// 64, 100 rows at H = 576, V = 49152 18.9, 19.2, 19.6, 20.1 -> 12.0, 12.4,
// 14.0, 16.8 us (the 256-row tiles of mf_gemm.hip); 128 rows of V = 50021
// 40.6 -> 18.3, of H = 2048, V = 128256 170 -> 140 (3.8 TB/s of table rows),
// so every call of up to 128 rows comes here.  The head of 9 rows at H = 960,
// V = 50021: 46.0 -> 20.9 us (the register-fed head it replaces); whole tails:
// 6 open rows of 64 at H = 576 36.6 -> 34.2 us, 70 of 700 at H = 1024,
// V = 90000 205 -> 168.
#include <hip/hip_runtime.h>

#include "mf_device.hpp"
#include "mf_head.hpp"
#include "mf_launch.hpp"

namespace mf {
namespace {

constexpr uint32_t kMmaWaves = 4;
constexpr uint32_t kCopyWaves = 4;
constexpr int kStreamThreads = static_cast<int>(64u * (kMmaWaves + kCopyWaves));
constexpr uint32_t kChunkF = 64;                     // features per chunk
constexpr uint32_t kRow = kChunkF * 2u;              // bytes of a row in a chunk
constexpr uint32_t kTileBlocksMax = 16;              // 16-token blocks per tile
constexpr uint32_t kTileMax = 16u * kTileBlocksMax;
constexpr uint32_t kWaveBlocks = kTileBlocksMax / kMmaWaves;
constexpr uint32_t kRingMax = 6;
constexpr uint32_t kLdsBytes = 160u * 1024u;

// The head's scores [slot][token], staged for the epilogue.  Rows of 260
// floats: the eight lanes of a slot read 128 bytes apart, the slots of a wave
// 4 banks apart, 16 bank groups in all.
constexpr uint32_t kScoreStride = kTileMax + 4u;
struct HeadStage {
  float g[kPanelRows][kScoreStride];
  float tn[kMmaWaves];
  uint32_t count[kMmaWaves][64];
  uint32_t src_row[kPanelRows];
  float src_norm[kPanelRows];
  float src_slack[kPanelRows];
};

struct StreamArgs {
  const uint16_t* a;      // A row r of M-tile t: a + t * a_tile + r * a_stride (halves)
  uint64_t a_tile;
  uint32_t a_stride;
  uint32_t m;             // A rows (linear: rows past the last re-read it)
  const uint16_t* emb;    // [V, H]
  uint32_t H;             // a multiple of 32
  uint32_t V;
  uint32_t nb;            // 16-token blocks per tile
  uint32_t tiles;
  uint32_t m_tiles;
  uint32_t ring;          // chunk buffers
  uint16_t* out;          // linear: FP16 [m, V]
  FallbackArgs head;      // head: slots and records
};

// Wait until at most n of this wave's vector memory operations are in flight
// (n <= 63; the instruction takes a constant).
template <int kLo, int kHi>
__device__ __forceinline__ void wait_in_flight(uint32_t n) {
  if constexpr (kLo == kHi) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLo) : "memory");
  } else {
    constexpr int kMid = (kLo + kHi + 1) / 2;
    if (n >= static_cast<uint32_t>(kMid)) {
      wait_in_flight<kMid, kHi>(n);
    } else {
      wait_in_flight<kLo, kMid - 1>(n);
    }
  }
}

__device__ __forceinline__ void ring_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// LDS byte offset of piece p (0..7) of row r of a chunk region.
__device__ __forceinline__ uint32_t piece_at(uint32_t r, uint32_t p) {
  return r * kRow + (p ^ ((r >> 1) & 7u)) * 16u;
}

// Barriers of a tile's epilogue, which the copy waves must join.
constexpr uint32_t kHeadBarriers = 2;

// The tile's window records: as head_records (mf_head.hpp), for tiles of nt
// tokens; a slot's score is the sum of A rows 2 j and 2 j + 1 (hi and lo).
__device__ __forceinline__ void stage_scores(HeadStage& e, const floatx4 (&acc)[4][kWaveBlocks],
                                             const floatx4 (&gram)[kWaveBlocks], uint32_t nt,
                                             uint32_t blocks) {
  const uint32_t lane = threadIdx.x % 64u;
  const uint32_t wave = threadIdx.x / 64u;
  const uint32_t col = lane % 16u;
  const uint32_t kb = lane / 16u;
  float tn = 0.0f;
#pragma unroll
  for (uint32_t j = 0; j < kWaveBlocks; ++j) {
    if (j >= blocks) break;
    const uint32_t t = (wave + kMmaWaves * j) * 16u + col;
    const uint32_t i = col % 4u;
    const float d = i == 0u ? gram[j][0] : (i == 1u ? gram[j][1] : (i == 2u ? gram[j][2] : gram[j][3]));
    // lanes of the Gram diagonal, tokens of the vocabulary
    if (col / 4u == kb && t < nt) tn = __builtin_fmaxf(tn, __fsqrt_rn(d) * (1.0f + 0x1p-7f));
#pragma unroll
    for (uint32_t rb = 0; rb < 4; ++rb) {
#pragma unroll
      for (uint32_t jj = 0; jj < 2; ++jj) {
        e.g[rb * 8u + 2u * kb + jj][t] = acc[rb][j][2 * jj] + acc[rb][j][2 * jj + 1];
      }
    }
  }
  // a NaN norm (a non-finite table row) propagates: the bound then fails the
  // finiteness test and the tile is rescored in full
  const bool any_nan = __ballot(tn != tn) != 0ull;
  const float tn_wave = wave_max(tn);
  if (lane == 0) e.tn[wave] = any_nan ? __builtin_nanf("") : tn_wave;
}

__device__ __forceinline__ void write_records(const FallbackArgs& f, HeadStage& e, uint32_t m0,
                                              uint32_t tile, uint32_t tiles, uint32_t tok0,
                                              uint32_t nt) {
  const uint32_t lane = threadIdx.x % 64u;
  const uint32_t wave = threadIdx.x / 64u;
  float tn_max = e.tn[0];
#pragma unroll
  for (uint32_t w = 1; w < kMmaWaves; ++w) {
    const float v = e.tn[w];
    tn_max = (tn_max != tn_max || v != v) ? __builtin_nanf("") : __builtin_fmaxf(tn_max, v);
  }
  constexpr uint32_t kSeg = kTileMax / 8u;  // tokens per lane
  const uint32_t sl = lane / 8u;
  const uint32_t j8 = lane % 8u;
  const uint32_t i = wave * 8u + sl;  // the lane's slot
  const uint32_t t0 = j8 * kSeg;
  float gv[kSeg];
  const float4* src = reinterpret_cast<const float4*>(&e.g[i][t0]);
#pragma unroll
  for (uint32_t q = 0; q < kSeg / 4u; ++q) {
    const float4 v = src[q];
    gv[4 * q] = v.x;
    gv[4 * q + 1] = v.y;
    gv[4 * q + 2] = v.z;
    gv[4 * q + 3] = v.w;
  }
  // tokens past the tile read as -inf / 0
  float gm = -__builtin_huge_valf();
  float sum = 0.0f;
#pragma unroll
  for (uint32_t k = 0; k < kSeg; ++k) {
    const bool in = t0 + k < nt;
    sum += in ? gv[k] : 0.0f;
    gv[k] = in ? gv[k] : -__builtin_huge_valf();
    gm = __builtin_fmaxf(gm, gv[k]);
  }
  // every score of the lane finite (a sum that overflows counts as not
  // finite: the tile is then rescored in full, which is exact too)
  const uint64_t fin_lanes = __ballot(__builtin_isfinite(sum));
  const bool slot_finite = ((fin_lanes >> (8u * sl)) & 0xFFull) == 0xFFull;
  const float G = lane8_max(gm);
  const float bs =
      __builtin_fmaf(tn_max, __builtin_fmaf(f.coef, e.src_norm[i], f.coef2), e.src_slack[i]);
  const float L = G - bs;
  uint32_t members = 0u;  // bit k: token t0 + k
#pragma unroll
  for (uint32_t k = 0; k < kSeg; ++k) members |= (gv[k] + bs >= L) ? (1u << k) : 0u;
  const uint32_t n = static_cast<uint32_t>(__popc(members));
  e.count[wave][lane] = n;
  wave_sync();
  const uint4 c0 = *reinterpret_cast<const uint4*>(&e.count[wave][8u * sl]);
  const uint4 c1 = *reinterpret_cast<const uint4*>(&e.count[wave][8u * sl + 4u]);
  const uint32_t cs[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
  uint32_t before = 0u;
  uint32_t total = 0u;
#pragma unroll
  for (uint32_t q = 0; q < 8; ++q) {
    before += q < j8 ? cs[q] : 0u;
    total += cs[q];
  }
  if (e.src_row[i] == kInvalidToken) return;
  const bool finite = slot_finite && bs < 0x1p100f;
  const bool ordinary = finite && total <= static_cast<uint32_t>(kTileMembers);
  TileRecord* rec = f.records + static_cast<uint64_t>(m0 + i) * tiles + tile;
  if (ordinary) {
    // the lane's members in ascending order, their scores read back
    uint32_t r = before;
    while (members != 0u) {
      const uint32_t k = static_cast<uint32_t>(__builtin_ctz(members));
      members &= members - 1u;
      const float gk = e.g[i][t0 + k];
      const uint32_t token = tok0 + t0 + k;
      rec->m[r] = TileMember{token, token, gk - bs, gk + bs};
      ++r;
    }
  }
  if (j8 == 0u) {
    rec->best_lower = L;
    rec->flags = ordinary ? 0u : (finite ? kTileRescoreAll | kTileCrowded : kTileRescoreAll);
    rec->min_token = tok0;
    rec->min_pos = tok0;
    rec->begin = tok0;
    rec->count = nt;
    rec->n_members = ordinary ? total : 0u;
    rec->upper_max = G + bs;
  }
}

template <uint32_t kMT, bool kHead>
__global__ __launch_bounds__(kStreamThreads) void stream_kernel(StreamArgs a) {
  static_assert(!kHead || kMT == 2u * kPanelRows, "hi and lo of a panel tile's slots");
  extern __shared__ __align__(16) unsigned char lds[];
  HeadStage& stage = *reinterpret_cast<HeadStage*>(lds);
  unsigned char* ring = lds + (kHead ? sizeof(HeadStage) : 0u);
  const uint32_t lane = threadIdx.x % 64u;
  const uint32_t wave = threadIdx.x / 64u;
  const uint32_t chunks = (a.H + kChunkF - 1u) / kChunkF;
  const uint32_t chunk_bytes = (kMT + 16u * a.nb) * kRow;
  const uint32_t items = a.tiles * a.m_tiles;
  const uint32_t mine = (items - blockIdx.x + gridDim.x - 1u) / gridDim.x;
  const uint32_t total = mine * chunks;  // chunks of this workgroup's stream

  if (wave >= kMmaWaves) {
    // copy i of a chunk: 8 rows; i < kMT / 8 A rows, then tokens.  This wave
    // takes copies cw, cw + 4, .. (past the last: the last again, so that
    // every copy wave has `per` in flight per chunk).
    constexpr uint32_t kPerMax = (kMT / 8u + kTileBlocksMax * 2u + kCopyWaves - 1u) / kCopyWaves;
    const uint32_t cw = wave - kMmaWaves;
    const uint32_t copies = kMT / 8u + 2u * a.nb;
    const uint32_t per = (copies + kCopyWaves - 1u) / kCopyWaves;
    const unsigned char* src[kPerMax];
    auto copy_of = [&](uint32_t u) {
      const uint32_t i = cw + kCopyWaves * u;
      return i < copies ? i : copies - 1u;
    };
    auto piece_of = [&](uint32_t r) { return (lane % 8u) ^ ((r >> 1) & 7u); };
    auto open_tile = [&](uint32_t item) {  // the lane's source of each copy at feature 0
      const uint32_t tile = item / a.m_tiles;
      const uint32_t mt = item - tile * a.m_tiles;
#pragma unroll
      for (uint32_t u = 0; u < kPerMax; ++u) {
        const uint32_t i = copy_of(u);
        const uint32_t r = 8u * i + lane / 8u;  // kMT is a multiple of 16
        if (i < kMT / 8u) {
          const uint32_t last = a.m - 1u - (kHead ? 0u : mt * kMT);
          const uint32_t row = (kHead || r <= last) ? r : last;
          src[u] = reinterpret_cast<const unsigned char*>(a.a + mt * a.a_tile +
                                                          static_cast<uint64_t>(row) * a.a_stride +
                                                          piece_of(r) * 8u);
        } else {
          const uint32_t b = r - kMT;
          const uint32_t t = tile * a.nb * 16u + b;
          src[u] = reinterpret_cast<const unsigned char*>(
              a.emb + static_cast<uint64_t>(t < a.V ? t : a.V - 1u) * a.H + piece_of(b) * 8u);
        }
      }
    };
    uint32_t item = blockIdx.x;  // position of the next chunk to issue
    uint32_t c = 0;
    uint32_t slot = 0;
    auto issue = [&]() {
      if (c == 0u) open_tile(item);
      unsigned char* buf = ring + slot * chunk_bytes;
      // a last half chunk: pieces past the row re-read the half before
      const bool cut = (c + 1u) * kChunkF > a.H;
#pragma unroll
      for (uint32_t u = 0; u < kPerMax; ++u) {
        if (u < per) {
          const uint32_t i = copy_of(u);
          const uint32_t r = 8u * i + lane / 8u;
          const uint32_t back = (cut && piece_of(r) >= 4u) ? 64u : 0u;
          burst_to_lds(src[u] + c * kRow - back, buf + i * 1024u);
        }
      }
      if (++c == chunks) {
        c = 0;
        item += gridDim.x;
      }
      if (++slot == a.ring) slot = 0;
    };
    const uint32_t ahead = a.ring - 1u;
    const uint32_t first = total < ahead ? total : ahead;
    for (uint32_t q = 0; q < first; ++q) issue();
    wait_in_flight<0, 63>((first - 1u) * per);
    ring_barrier();  // chunk 0 in LDS
    uint32_t left = chunks;
    for (uint32_t q = 0; q < total; ++q) {
      // the MFMA waves work on chunk q; chunk q - 1's buffer is free
      if (q + ahead < total) issue();
      if (q + 1u < total) {
        const uint32_t last = q + ahead < total ? q + ahead : total - 1u;
        wait_in_flight<0, 63>((last - (q + 1u)) * per);
      }
      ring_barrier();  // chunk q + 1 in LDS, chunk q read
      if (--left == 0u) {
        left = chunks;
        if constexpr (kHead) {
          for (uint32_t k = 0; k < kHeadBarriers; ++k) ring_barrier();
        }
      }
    }
    return;
  }

  // MFMA waves: wave w takes the tile's 16-token blocks w, w + 4, ..
  constexpr uint32_t kRb = kMT / 16u;
  const uint32_t col = lane % 16u;
  const uint32_t kb = lane / 16u;
  ring_barrier();
  uint32_t slot = 0;
  for (uint32_t item = blockIdx.x; item < items; item += gridDim.x) {
    const uint32_t tile = item / a.m_tiles;
    const uint32_t mt = item - tile * a.m_tiles;
    const uint32_t tok0 = tile * a.nb * 16u;
    const uint32_t nt = a.V - tok0 < a.nb * 16u ? a.V - tok0 : a.nb * 16u;
    const uint32_t blocks = a.nb > wave ? (a.nb - wave + kMmaWaves - 1u) / kMmaWaves : 0u;
    if constexpr (kHead) {  // read after the chunk barriers below
      if (threadIdx.x < kPanelRows) {
        const FallbackArgs& f = a.head;
        const uint32_t i = mt * kPanelRows + threadIdx.x;
        const uint32_t at = i < f.m ? i : f.m - 1u;
        const uint32_t row = f.slot_row[at];
        const uint32_t r = i < f.m ? row : kInvalidToken;
        stage.src_row[threadIdx.x] = r;
        stage.src_norm[threadIdx.x] = r != kInvalidToken ? f.slot_norm[at] : 0.0f;
        stage.src_slack[threadIdx.x] = r != kInvalidToken ? f.slot_slack[at] : 0.0f;
        if (tile == 0u && r != kInvalidToken && f.fb_map != nullptr) f.fb_map[r] = i;
      }
    }
    floatx4 acc[kRb][kWaveBlocks];
    floatx4 gram[kWaveBlocks];
#pragma unroll
    for (uint32_t j = 0; j < kWaveBlocks; ++j) {
      gram[j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (uint32_t rb = 0; rb < kRb; ++rb) acc[rb][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    for (uint32_t c = 0; c < chunks; ++c) {
      const unsigned char* abuf = ring + slot * chunk_bytes;
      const unsigned char* bbuf = abuf + kMT * kRow;
#pragma unroll
      for (uint32_t s = 0; s < 2u; ++s) {
        if (c * kChunkF + 32u * s >= a.H) break;
        const uint32_t p = 4u * s + kb;
        half8_t af[kRb];
#pragma unroll
        for (uint32_t rb = 0; rb < kRb; ++rb) {
          af[rb] = *reinterpret_cast<const half8_t*>(abuf + piece_at(16u * rb + col, p));
        }
#pragma unroll
        for (uint32_t j = 0; j < kWaveBlocks; ++j) {
          if (j >= blocks) break;
          const half8_t bf = *reinterpret_cast<const half8_t*>(
              bbuf + piece_at((wave + kMmaWaves * j) * 16u + col, p));
          if constexpr (kHead) {
            gram[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf, bf, gram[j], 0, 0, 0);
          }
#pragma unroll
          for (uint32_t rb = 0; rb < kRb; ++rb) {
            acc[rb][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[rb], bf, acc[rb][j], 0, 0, 0);
          }
        }
      }
      if (++slot == a.ring) slot = 0;
      ring_barrier();
    }
    if constexpr (kHead) {
      stage_scores(stage, acc, gram, nt, blocks);
      ring_barrier();
      write_records(a.head, stage, mt * kPanelRows, tile, a.tiles, tok0, nt);
      ring_barrier();  // the stage is free for the next tile
    } else {
      // D of block (rb, j): lane l holds rows 4 (l / 16) + i, column l % 16
#pragma unroll
      for (uint32_t j = 0; j < kWaveBlocks; ++j) {
        if (j >= blocks) break;
        const uint32_t t = (wave + kMmaWaves * j) * 16u + col;
        if (t >= nt) continue;
#pragma unroll
        for (uint32_t rb = 0; rb < kRb; ++rb) {
#pragma unroll
          for (uint32_t i = 0; i < 4u; ++i) {
            const uint32_t row = mt * kMT + 16u * rb + 4u * kb + i;
            if (row < a.m) {
              a.out[static_cast<uint64_t>(row) * a.V + tok0 + t] = float_to_half_rne(acc[rb][j][i]);
            }
          }
        }
      }
    }
  }
}

template <uint32_t kMT, bool kHead>
hipError_t launch_stream(StreamArgs a, uint32_t groups, hipStream_t stream) {
  a.tiles = stream_tiles(a.V, a.nb);
  const uint32_t stage = kHead ? static_cast<uint32_t>(sizeof(HeadStage)) : 0u;
  const uint32_t chunk = (kMT + 16u * a.nb) * kRow;
  const uint32_t fit = (kLdsBytes - stage) / chunk;
  a.ring = fit < kRingMax ? fit : kRingMax;
  static_assert((kLdsBytes - (kHead ? sizeof(HeadStage) : 0u)) / ((kMT + kTileMax) * kRow) >= 2u,
                "two chunks fit");
  const uint64_t items = static_cast<uint64_t>(a.tiles) * a.m_tiles;
  if (items > 0xFFFFFFFFull || items * ((a.H + kChunkF - 1u) / kChunkF) > 0xFFFFFFFFull) {
    return hipErrorInvalidValue;
  }
  const uint32_t cus = groups > 0 ? groups : kStreamCUs;
  const dim3 grid(items < cus ? static_cast<uint32_t>(items) : cus);
  hipLaunchKernelGGL((stream_kernel<kMT, kHead>), grid, dim3(kStreamThreads),
                     stage + a.ring * chunk, stream, a);
  return hipGetLastError();
}

}  // namespace

// Blocks of 16 tokens per tile: the fewest rounds of 256 tiles of at most 16
// blocks, then tiles just large enough for them (V = 49152: 256 tiles of 12
// blocks; 50021: 241 of 13; 128256: 501 of 16, two rounds), of at least two
// blocks (a tile's A rows come with it).  Coarse: at least the 12 blocks of
// the table pass's tiles (fewer records for a small vocabulary).  A fixed
// number of compute units: the records' layout must not depend on where it
// is sized.
uint32_t stream_tile_blocks(uint32_t vocab, bool coarse) {
  const uint64_t blocks = (static_cast<uint64_t>(vocab) + 15u) / 16u;
  const uint64_t rounds = (blocks + kStreamCUs * kTileBlocksMax - 1u) / (kStreamCUs * kTileBlocksMax);
  const uint64_t nb = (blocks + kStreamCUs * rounds - 1u) / (kStreamCUs * rounds);
  const uint64_t least = coarse ? kHeadTileTokens / 16u : 2u;
  return static_cast<uint32_t>(nb > least ? nb : least);
}
uint32_t stream_tiles(uint32_t vocab, uint32_t blocks) {
  return static_cast<uint32_t>((static_cast<uint64_t>(vocab) + 16u * blocks - 1u) / (16u * blocks));
}

hipError_t launch_stream_head(const FallbackArgs& f, uint32_t blocks, hipStream_t stream) {
  if (f.m == 0) return hipSuccess;
  if (f.H % 64 != 0 || f.panel == nullptr || blocks == 0 || blocks > kTileBlocksMax) {
    return hipErrorInvalidValue;
  }
  StreamArgs a{};
  a.a = f.panel;
  a.a_tile = panel_tile_bytes(f.H) / 2u;
  a.a_stride = f.H + kPanelPad;
  a.m = f.m;
  a.emb = f.emb;
  a.H = f.H;
  a.V = f.V;
  a.nb = blocks;
  a.m_tiles = panel_tiles(f.m);
  a.head = f;
  return launch_stream<2u * kPanelRows, true>(a, f.groups, stream);
}

hipError_t launch_stream_linear(const ProjArgs& p, uint32_t groups, hipStream_t stream) {
  if (p.H % 32 != 0 || p.H == 0 || p.m == 0 || p.m > kStreamRowsMax || p.V == 0 ||
      p.a16 == nullptr || p.emb == nullptr || p.out_f16 == nullptr ||
      reinterpret_cast<uintptr_t>(p.a16) % 16u != 0 || reinterpret_cast<uintptr_t>(p.emb) % 16u != 0) {
    return hipErrorInvalidValue;
  }
  StreamArgs a{};
  a.a = p.a16;
  a.a_stride = p.H;
  a.m = p.m;
  a.emb = p.emb;
  a.H = p.H;
  a.V = p.V;
  a.nb = stream_tile_blocks(p.V, false);
  a.m_tiles = 1;
  a.out = p.out_f16;
  if (p.m <= 16u) return launch_stream<16, false>(a, groups, stream);
  if (p.m <= 32u) return launch_stream<32, false>(a, groups, stream);
  if (p.m <= 64u) return launch_stream<64, false>(a, groups, stream);
  return launch_stream<128, false>(a, groups, stream);
}

}  // namespace mf
