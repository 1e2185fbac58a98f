// The dense head: one pass over the FP16 table in 192-token tiles that
// scores every row of a panel against every token of the tile with MFMA, and
// keeps, per (row, tile), the window record of the tokens the row allows.
//
// Its rows (slots): the unrestricted rows of the call (all tokens allowed),
// then the restricted rows with long ascending lists that the norm launch
// marked kRowDense.  For such a row the gather would read one 4 KiB table
// row per candidate (at H = 2048, 1.5 M candidates are 6.5 GB); the dense
// head reads each table row once per panel of 256 slots and pays in MFMA
// work instead (2 H flops per slot and token).
//
// Workgroup: a panel of 256 slots (16 blocks of 16) x one tile of 12 token
// blocks, twelve waves.  Eight MFMA waves, two a SIMD, so that one's MFMAs run
// under the other's LDS reads: wave w (0-7) takes the row blocks 4 i + w % 4
// and the six token blocks of half w / 4 (4 x 6 MFMA blocks,
// v_mfma_f32_16x16x32_f16); waves 8-11 issue the copies (a wave issuing
// copies stalls while the address unit is busy, and an MFMA wave would idle
// with it).  K runs in chunks of 64 features (whole 128-byte lines): a chunk's
// A rows (the slots' FP16 hi of z = x * w, from L2) in four units of 64 rows
// and its B rows (the tile's table rows, from HBM) are copied straight into LDS
// (global_load_lds, 16 bytes per lane), into rings of two chunks and a unit
// and of three chunks; one barrier per chunk, where every MFMA wave has its
// last fragments in registers.  The 16-byte pieces of a row are XOR-swizzled
// by the row's bits 1-3, so the 16 lanes one read cycle serves meet 16 bank
// groups.  The MFMA waves also sum the squares of the table fragments they read
// (FP32, any order), which gives the token norms of the bounds.
// One panel (51 open and 205 listed rows) at H = 2048, V = 128256, three
// tiles on most compute units: 198 -> 174 us (from 32-feature steps, 64 bytes a
// row, in four MFMA waves); bound by the copies as the projection GEMM (1.4 us a
// chunk) and by the epilogue and first copies of each tile, about 14 us.
//
// Epilogue per tile: the slot's allowed tokens of the tile come from the
// norm launch's span index (a 192-bit mask and the list position of the
// first id), copied into LDS ahead of the tile's chunks; per slot the best
// lower bound over allowed tokens, the members (fl(g + b) >= L) and one
// TileRecord in the MFMA head's format (list positions for restricted rows,
// token ids for unrestricted ones).
//
// Workgroups: one per compute unit.  Each computes the slot list itself (a
// prefix over the rows' kinds), so P = ceil(slots / 256) panels of equal
// size (to one slot); row blocks past a panel's slots get no MFMA.  The
// compute units of an XCD (blockIdx % 8) form groups of P workgroups that
// run the same run of tiles, one panel each, so the table tiles of a group
// are read from HBM once and from the XCD's L2 by the other panels.
#include <hip/hip_runtime.h>

#include "mf_device.hpp"
#include "mf_launch.hpp"

namespace mf {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kMmaWaves = 8;
constexpr int kCopyWaves = 4;
constexpr int kWaves = kMmaWaves + kCopyWaves;
constexpr int kThreads = kWaves * kWave;
constexpr int kRBw = 4;     // row blocks per MFMA wave
constexpr int kTBw = 6;     // token blocks per MFMA wave
constexpr int kNormBw = 2;  // token blocks whose norms an MFMA wave forms, at most
constexpr uint32_t kKC = 64;          // features per chunk
constexpr uint32_t kRow = kKC * 2u;   // bytes of a row in a chunk
// the rings: A rows in units of 64 (one row block of each MFMA wave), two
// chunks and a unit; the tile's table rows, three chunks
constexpr uint32_t kAUnits = 4;
constexpr uint32_t kASlots = 2u * kAUnits + 1u;
constexpr uint32_t kAUnitRows = kDensePanelSlots / kAUnits;
constexpr uint32_t kAUnitBytes = kAUnitRows * kRow;
constexpr uint32_t kBSlots = 3;
constexpr uint32_t kBBytes = kHeadTileTokens * kRow;
constexpr uint32_t kRingBytes = kASlots * kAUnitBytes + kBSlots * kBBytes;
constexpr int kACopies = static_cast<int>(kAUnitBytes / 1024u / kCopyWaves);  // 1 KiB copies per wave
constexpr int kBCopies = static_cast<int>(kBBytes / 1024u / kCopyWaves);
static_assert(kACopies == 2 && kBCopies == 6, "copy split");
// copies per wave: what is brought ahead of the chunk before (a unit of A,
// the table rows), and the rest of a chunk
constexpr int kAhead = kACopies + kBCopies;
constexpr int kRest = static_cast<int>(kAUnits - 1u) * kACopies;
// epilogue rows in the rings' area: [slot][33] arrays of the lanes' values
// (two of floats, one of bytes), then the tile's records staged for the
// store
constexpr uint32_t kEpiRow = 33;
constexpr uint32_t kEpiRowsBytes = kDensePanelSlots * kEpiRow * 4u;
constexpr uint32_t kEpiBlockBytes = (kDensePanelSlots * kEpiRow + 15u) / 16u * 16u;  // bytes
static_assert(2u * kEpiRowsBytes + kEpiBlockBytes + kDensePanelSlots * 96u <= kRingBytes,
              "epilogue rows and staged records in the rings");
static_assert(2 * kTBw == static_cast<int>(kHeadTileTokens / 16u) &&
                  4 * kRBw * 16 == static_cast<int>(kDensePanelSlots),
              "tile and panel");

enum : uint32_t { kSlotNone = 0u, kSlotAll = 1u, kSlotList = 2u };

struct DenseShared {
  uint32_t slot_row[kDensePanelSlots];
  float slot_norm[kDensePanelSlots];
  float slot_slack[kDensePanelSlots];
  uint32_t slot_kind[kDensePanelSlots];
  uint4 span[kDensePanelSlots][2];  // {m0,m1,m2,lo},{m3,m4,m5,cnt}
  float tn[kMmaWaves];
  uint32_t wave_sum[kWaves];
};

__host__ __device__ constexpr uint32_t dense_lds_bytes() {
  return kRingBytes + static_cast<uint32_t>(sizeof(DenseShared));
}

static_assert(dense_lds_bytes() <= 160u * 1024u, "LDS");

// LDS byte offset of piece p (0..7) of row r of a ring slot: the 16 lanes one
// ds_read_b128 cycle serves meet 16 bank groups
__device__ __forceinline__ uint32_t swz(uint32_t r) { return (r >> 1) & 7u; }
__device__ __forceinline__ uint32_t piece_at(uint32_t r, uint32_t p) { return r * kRow + (p ^ swz(r)) * 16u; }

// The slot list of the launch: unrestricted rows first (fb_rows order), then
// the kRowDense rows in row order; panel p of P takes slots [p0, p0 + n)
// with p0 = p S / P (S slots), so the panels differ by one slot at most.
// Fills this panel's slot table.
__device__ void dense_slots(const DenseArgs& a, DenseShared& sh, uint32_t p0, uint32_t n,
                            bool map) {
  const uint32_t tid = threadIdx.x;
  const uint32_t lane = tid % kWave;
  const uint32_t wave = tid / kWave;
  const uint32_t per = (a.rows + kThreads - 1) / kThreads;
  const uint32_t r0 = tid * per < a.rows ? tid * per : a.rows;
  const uint32_t r1 = r0 + per < a.rows ? r0 + per : a.rows;
  uint32_t local = 0u;
  for (uint32_t r = r0; r < r1; ++r) local += (a.row_meta[r].kind & kRowDense) ? 1u : 0u;
  uint32_t incl = local;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t o = static_cast<uint32_t>(__shfl_up(static_cast<int>(incl), d));
    if (static_cast<int>(lane) >= d) incl += o;
  }
  if (tid < kDensePanelSlots) sh.slot_kind[tid] = kSlotNone;
  if (lane == kWave - 1) sh.wave_sum[wave] = incl;
  __syncthreads();
  uint32_t before = incl - local;
#pragma unroll
  for (uint32_t w = 0; w < kWaves; ++w) before += w < wave ? sh.wave_sum[w] : 0u;
  // unrestricted slots of this panel (a listed row that is not unrestricted,
  // or not a row, gets no slot work)
  {
    const uint32_t gs = p0 + tid;
    if (tid < n && gs < a.fb_m) {
      const uint32_t r = a.fb_rows[gs];
      if (r < a.rows && (a.row_meta[r].kind & kRowUnrestricted)) {
        sh.slot_row[tid] = r;
        sh.slot_kind[tid] = kSlotAll;
      }
    }
  }
  // dense rows of this panel
  uint32_t k = a.fb_m + before;
  for (uint32_t r = r0; r < r1; ++r) {
    if (a.row_meta[r].kind & kRowDense) {
      if (k >= p0 && k < p0 + n) {
        sh.slot_row[k - p0] = r;
        sh.slot_kind[k - p0] = kSlotList;
      }
      ++k;
    }
  }
  __syncthreads();
  if (tid < kDensePanelSlots) {
    const uint32_t kind = sh.slot_kind[tid];
    const uint32_t r = kind != kSlotNone ? sh.slot_row[tid] : 0u;
    sh.slot_norm[tid] = kind != kSlotNone ? a.row_norm[r] : 0.0f;
    sh.slot_slack[tid] = kind != kSlotNone ? a.row_slack[r] : 0.0f;
    if (kind == kSlotNone) sh.slot_row[tid] = 0u;  // a valid row for the copies
    if (map && kind != kSlotNone) a.fb_map[r] = p0 + tid;
  }
  __syncthreads();
}

// Wait until at most kN of this copy wave's copies are in flight.
template <int kN>
__device__ __forceinline__ void wait_copies() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kN) : "memory");
}

// A workgroup barrier without __syncthreads' release fence, which would wait
// for every LDS-DMA copy in flight (vector memory count 0) and empty the
// pipeline.  The wave's own LDS operations are complete when it arrives.
__device__ __forceinline__ void step_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__global__ __launch_bounds__(kThreads) void dense_kernel(DenseArgs a) {
  extern __shared__ __align__(16) unsigned char dyn[];
  DenseShared& sh = *reinterpret_cast<DenseShared*>(dyn + kRingBytes);
  const uint32_t tid = threadIdx.x;
  const uint32_t lane = tid % kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const bool copier = wave >= static_cast<uint32_t>(kMmaWaves);
  const uint32_t cw = wave % kCopyWaves;  // copy wave index (copy waves)
  const uint32_t wm = wave % 4u;  // row block of each unit (MFMA waves)
  const uint32_t wn = (wave / 4u) % 2u;  // token half (MFMA waves)
  const uint32_t col = lane % 16u;
  const uint32_t kb = lane / 16u;
  // workgroup -> (group, panel): the compute units of one XCD in groups of
  // P consecutive local indices.  The slot count is computed first with
  // panel 0's table (every workgroup needs it).
  const uint32_t xcds = 8u;
  const uint32_t per_xcd = gridDim.x / xcds;
  const uint32_t x = blockIdx.x % xcds;
  const uint32_t l = blockIdx.x / xcds;
  uint32_t n_slots;
  {
    // the count does not depend on the panel; the table of the true panel
    // is built below
    const uint32_t per = (a.rows + kThreads - 1) / kThreads;
    const uint32_t r0 = tid * per < a.rows ? tid * per : a.rows;
    const uint32_t r1 = r0 + per < a.rows ? r0 + per : a.rows;
    uint32_t local = 0u;
    for (uint32_t r = r0; r < r1; ++r) local += (a.row_meta[r].kind & kRowDense) ? 1u : 0u;
    local = wave_sum_u32(local);
    if (lane == 0) sh.wave_sum[wave] = local;
    __syncthreads();
    n_slots = a.fb_m;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) n_slots += sh.wave_sum[w];
    __syncthreads();
  }
  const uint32_t P = (n_slots + kDensePanelSlots - 1) / kDensePanelSlots;
  if (P == 0u || P > per_xcd) return;  // the launcher bounds P by per_xcd
  const uint32_t gpx = per_xcd / P;
  if (l >= gpx * P) return;
  const uint32_t panel = l % P;
  const uint32_t p0 = panel * n_slots / P;
  const uint32_t pn = (panel + 1u) * n_slots / P - p0;
  // row blocks with slots; waves wm take blocks 4 i + wm, i < nact
  const uint32_t nrb = (pn + 15u) / 16u;
  const uint32_t nact = nrb > wm ? (nrb - wm + 3u) / 4u : 0u;
  const uint32_t grp = x * gpx + l / P;
  const uint32_t groups = xcds * gpx;
  const uint32_t tiles = a.ranges;
  const uint32_t t_begin = static_cast<uint32_t>(static_cast<uint64_t>(tiles) * grp / groups);
  const uint32_t t_end = static_cast<uint32_t>(static_cast<uint64_t>(tiles) * (grp + 1u) / groups);
  dense_slots(a, sh, p0, pn, grp == 0u);
  const uint32_t H = a.H;
  const uint32_t chunks = (H + kKC - 1u) / kKC;
  unsigned char* const bring = dyn + kASlots * kAUnitBytes;
  // The tile's LDS epilogue areas (the rings, free after the K loop):
  // per-lane values of each slot in rows of 33 words (word 16 half + column
  // of slot s's row, padded so the four slots of one write sit on different
  // banks), then the tile's records, staged for the store.
  float* gl1 = reinterpret_cast<float*>(dyn);                          // best
  float* gl2 = reinterpret_cast<float*>(dyn + kEpiRowsBytes);          // second best
  uint8_t* glj = dyn + 2u * kEpiRowsBytes;  // token block of the best
  TileRecord* stage_rec = reinterpret_cast<TileRecord*>(dyn + 2u * kEpiRowsBytes + kEpiBlockBytes);
  // the staged records out, 16 bytes per thread and step (each record is
  // contiguous in global memory); no wait for these stores before the next
  // tile, only for the LDS reads
  auto store_records = [&](uint32_t tile) {
    constexpr uint32_t kPieces = sizeof(TileRecord) / 16u;
    const uint4* from = reinterpret_cast<const uint4*>(stage_rec);
    uint32_t u0 = tid;
    asm volatile("" : "+v"(u0));
    for (uint32_t u = u0; u < kDensePanelSlots * kPieces; u += kThreads) {
      const uint32_t s = u / kPieces;
      if (sh.slot_kind[s] == kSlotNone) continue;
      uint4* to = reinterpret_cast<uint4*>(a.records + (static_cast<uint64_t>(p0) + s) * tiles + tile);
      to[u % kPieces] = from[u];
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  // The copy waves: every tile's chunks, then the barriers of the MFMA
  // waves' epilogue.  (Separate loops for the two kinds of waves, so that
  // neither holds the other's registers.)
  auto copy_tiles = [&]() {
    // per-lane copy sources of a copy wave: copy i of unit u brings A rows
    // 64 u + 8 (cw + 4 i) .., lane l row l / 8 of them, LDS piece l % 8; the
    // span records (2 copies of 32 slots)
    uint32_t aoff[kAUnits][kACopies];
#pragma unroll
    for (uint32_t u = 0; u < kAUnits; ++u) {
#pragma unroll
      for (int i = 0; i < kACopies; ++i) {
        const uint32_t r = kAUnitRows * u + 8u * (cw + kCopyWaves * i) + lane / 8u;
        aoff[u][i] = sh.slot_row[r] * H + (((lane % 8u) ^ swz(r)) * 8u);
      }
    }
    uint32_t srow[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint32_t s = ((cw * 2u + j) * kWave + lane) / 2u;
      srow[j] = sh.slot_kind[s] == kSlotList ? sh.slot_row[s] : 0u;
    }
    // (rows 8 n + lane / 8 with the same lane share their swizzle up to n's
    // parity; a piece past a last half chunk re-reads the half before)
    const uint32_t piece0 = (lane % 8u) ^ swz(8u * cw + lane / 8u);
    for (uint32_t tile = t_begin; tile < t_end; ++tile) {
      const uint32_t tok0 = tile * kHeadTileTokens;
      const uint32_t nt = a.V - tok0 < kHeadTileTokens ? a.V - tok0 : kHeadTileTokens;
      {
        uint4* dst = &sh.span[0][0];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const uint32_t idx = (cw * 2u + j) * kWave + lane;
          const uint4* src = a.spans + (static_cast<uint64_t>(tile) * a.rows + srow[j]) * 2u + (idx % 2u);
          burst_to_lds(src, dst + (cw * 2u + j) * kWave);
        }
      }
      const uint16_t* tbase = a.emb + static_cast<uint64_t>(tok0) * H;
      uint32_t boff[kBCopies];
#pragma unroll
      for (int i = 0; i < kBCopies; ++i) {
        const uint32_t t = 8u * (cw + kCopyWaves * i) + lane / 8u;
        const uint32_t tc = t < nt ? t : nt - 1u;
        boff[i] = tc * H + (((lane % 8u) ^ swz(t)) * 8u);
      }
      // the features of chunk c at this lane's pieces
      auto feature = [&](uint32_t c) {
        return c * kKC - (c * kKC + piece0 * 8u >= H ? 32u : 0u);
      };
      uint32_t aslot = 0, bslot = 0;  // the next unit's and chunk's
      auto issue_a = [&](uint32_t c, uint32_t u) {
        unsigned char* buf = dyn + aslot * kAUnitBytes;
        const uint32_t f = feature(c);
#pragma unroll
        for (int i = 0; i < kACopies; ++i) {
          const uint32_t off = u == 0u ? aoff[0][i] : (u == 1u ? aoff[1][i] : (u == 2u ? aoff[2][i] : aoff[3][i]));
          burst_to_lds(a.z_hi + off + f, buf + (cw + kCopyWaves * i) * 1024u);
        }
        if (++aslot == kASlots) aslot = 0u;
      };
      auto issue_ahead = [&](uint32_t c) {
        issue_a(c, 0u);
        unsigned char* buf = bring + bslot * kBBytes;
        const uint32_t f = feature(c);
#pragma unroll
        for (int i = 0; i < kBCopies; ++i) {
          burst_to_lds(tbase + boff[i] + f, buf + (cw + kCopyWaves * i) * 1024u);
        }
        if (++bslot == kBSlots) bslot = 0u;
      };
      auto issue_rest = [&](uint32_t c) {
        issue_a(c, 1u);
        issue_a(c, 2u);
        issue_a(c, 3u);
      };
      // two chunks and the part of a third in flight (the launcher checks
      // that there are three); then per chunk c, once chunk c + 1 has landed and
      // every MFMA wave has read chunk c, what its slots make room for
      issue_ahead(0u);
      issue_rest(0u);
      issue_ahead(1u);
      issue_rest(1u);
      issue_ahead(2u);
      wait_copies<2 * kAhead + kRest>();
      step_barrier();  // chunk 0 in LDS
      for (uint32_t c = 0; c < chunks; ++c) {
        if (c + 2u < chunks) {
          wait_copies<kAhead>();
        } else {
          wait_copies<0>();
        }
        step_barrier();  // chunk c + 1 in LDS, chunk c read by every MFMA wave
        if (c + 2u < chunks) issue_rest(c + 2u);
        if (c + 3u < chunks) issue_ahead(c + 3u);
      }
      // the MFMA waves' epilogue phases (the same barriers)
      __syncthreads();
      __syncthreads();
      __syncthreads();
      store_records(tile);
    }
  };
  // The MFMA waves (threads 0 .. 255 also stand for the panel's slots), with
  // NACT of the wave's row blocks holding slots (a variant per count, so the loop has no branch
  // around an MFMA).
  auto mfma_tiles = [&]<int NACT>() {
    for (uint32_t tile = t_begin; tile < t_end; ++tile) {
      const uint32_t tok0 = tile * kHeadTileTokens;
      const uint32_t nt = a.V - tok0 < kHeadTileTokens ? a.V - tok0 : kHeadTileTokens;
      floatx4 acc[kRBw][kTBw];
#pragma unroll
      for (int i = 0; i < kRBw; ++i) {
#pragma unroll
        for (int j = 0; j < kTBw; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
      }
      // per lane: the sums of squares of its features of the tokens of the
      // wave's norm blocks (token blocks wm, wm + 4 of its half)
      float tsq[kNormBw] = {0.0f, 0.0f};
      uint32_t as = 0, bs = 0;  // the slots of the chunk's first unit and table rows
      half8_t fa[kRBw], fb[kTBw];
      auto read_half = [&](uint32_t h) {
        const uint32_t p = 4u * h + kb;
        const unsigned char* bbuf = bring + bs * kBBytes;
#pragma unroll
        for (int j = 0; j < kTBw; ++j) {
          fb[j] = *reinterpret_cast<const half8_t*>(bbuf + piece_at((wn * kTBw + j) * 16u + col, p));
        }
#pragma unroll
        for (int i = 0; i < NACT; ++i) {
          const uint32_t slot = as + i < kASlots ? as + i : as + i - kASlots;
          fa[i] = *reinterpret_cast<const half8_t*>(dyn + slot * kAUnitBytes + piece_at(16u * wm + col, p));
        }
      };
      auto multiply = [&]() {
#pragma unroll
        for (int i = 0; i < NACT; ++i) {
#pragma unroll
          for (int j = 0; j < kTBw; ++j) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[i], fb[j], acc[i][j], 0, 0, 0);
          }
        }
#pragma unroll
        for (int j = 0; j < kTBw; ++j) {
          if (static_cast<uint32_t>(j % 4) == wm) {  // (wave-uniform)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float v = static_cast<float>(fb[j][e]);
              tsq[j / 4] = __builtin_fmaf(v, v, tsq[j / 4]);
            }
          }
        }
      };
      step_barrier();  // chunk 0 in LDS
      for (uint32_t c = 0; c < chunks; ++c) {
        read_half(0u);
        multiply();
        read_half(1u);
        step_barrier();  // this wave's reads of chunk c have arrived
        if ((as += kAUnits) >= kASlots) as -= kASlots;
        if (++bs == kBSlots) bs = 0u;
        if (c * kKC + 32u < H) multiply();
      }
      // (after the last barrier nothing reads or writes the rings)

      // token norms: lanes c, c + 16, c + 32, c + 48 hold the four K
      // quarters of column c's sum; a NaN norm (non-finite table row)
      // propagates
      {
        // (the lane's indices made opaque here, so that the compiler forms
        // them after the K loop instead of holding them through it)
        uint32_t el = lane;
        asm volatile("" : "+v"(el));
        const uint32_t ecol = el % 16u;
        const uint32_t t0 = (wn * kTBw + wm) * 16u + ecol;
        const int up16 = static_cast<int>((el ^ 16u) * 4u);
        const int up32 = static_cast<int>((el ^ 32u) * 4u);
        float tn_local = 0.0f;
        bool tn_nan = false;
#pragma unroll
        for (int j = 0; j < kNormBw; ++j) {
          float q = tsq[j];
          q += __int_as_float(__builtin_amdgcn_ds_bpermute(up16, __float_as_int(q)));
          q += __int_as_float(__builtin_amdgcn_ds_bpermute(up32, __float_as_int(q)));
          const uint32_t t = t0 + 64u * static_cast<uint32_t>(j);
          if (el < 16u && t < nt && wm + 4u * static_cast<uint32_t>(j) < kTBw) {
            const float v = __fsqrt_rn(q) * (1.0f + 0x1p-7f);
            tn_nan |= v != v;
            tn_local = __builtin_fmaxf(tn_local, v);
          }
        }
        const bool any_nan = __ballot(tn_nan) != 0ull;
        const float m = wave_max(tn_local);
        if (lane == 0) sh.tn[wave] = any_nan ? __builtin_nanf("") : m;
      }
      // the allowed words of every slot in its span record: unrestricted
      // slots allow the tile's tokens below nt, empty slots nothing
      // (thread tid's slot index made opaque here for the same reason)
      uint32_t es = tid;
      asm volatile("" : "+v"(es));
      if (es < kDensePanelSlots) {
        const uint32_t kind = sh.slot_kind[es];
        if (kind != kSlotList) {
          uint32_t w[6];
#pragma unroll
          for (int k = 0; k < 6; ++k) {
            const uint32_t lo = k * 32u;
            w[k] = kind == kSlotNone ? 0u
                   : (nt >= lo + 32u ? 0xFFFFFFFFu : (nt > lo ? (1u << (nt - lo)) - 1u : 0u));
          }
          sh.span[es][0] = uint4{w[0], w[1], w[2], tok0};
          sh.span[es][1] = uint4{w[3], w[4], w[5], kind == kSlotNone ? 0u : nt};
        }
      }
      __syncthreads();
      // lane bases: slot (i, q) of this lane is sbase + 64 i + q (opaque to
      // the compiler, so that the epilogue's addresses are formed here and not
      // hoisted out of the tile loop, where they would outlive the registers)
      uint32_t sbase = wm * 16u + 4u * kb;
      asm volatile("" : "+v"(sbase));
      const uint4* spn = &sh.span[sbase][wn];
      const uint32_t sel0 = 1u << col;
      const uint32_t sel1 = 1u << (16u + col);
      const uint32_t lw = sbase * kEpiRow + wn * 16u + col;  // this lane's word of slot sbase
      // per slot and MFMA lane: the best and second best allowed scores of
      // the lane's six tokens and the block of the best (the best is NaN when
      // one of its allowed scores is not finite); the row blocks past the
      // panel's slots hold none of its slots
#pragma unroll
      for (int i = 0; i < NACT; ++i) {
        uint4 w4[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) w4[q] = spn[(64 * i + q) * 2];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t w[3] = {w4[q].x, w4[q].y, w4[q].z};
          // arithmetic form (one condition per select, no lane-mask logic):
          // va = the score or -inf, vb - vb is NaN exactly when an allowed score is
          // not finite
          float m1 = -__builtin_huge_valf();
          float m2 = -__builtin_huge_valf();
          float badacc = 0.0f;
          uint32_t j1 = 0u;
#pragma unroll
          for (int j = 0; j < kTBw; ++j) {
            const bool allowed = (w[j / 2] & (j % 2 == 0 ? sel0 : sel1)) != 0u;
            const float v = acc[i][j][q];
            const float va = allowed ? v : -__builtin_huge_valf();
            const float vb = allowed ? v : 0.0f;
            badacc += vb - vb;
            m2 = __builtin_fmaxf(m2, __builtin_fminf(m1, va));
            j1 = va > m1 ? static_cast<uint32_t>(j) : j1;
            m1 = __builtin_fmaxf(m1, va);
          }
          gl1[lw + (64 * i + q) * kEpiRow] = badacc != badacc ? __builtin_nanf("") : m1;
          gl2[lw + (64 * i + q) * kEpiRow] = m2;
          glj[lw + (64 * i + q) * kEpiRow] = static_cast<uint8_t>(j1);
        }
      }
      __syncthreads();
      // the slot's record (thread s), written into its LDS stage.  G = the
      // best allowed score, b the bound, L = fl(G - b); the members are the
      // lane bests with fl(g + b) >= L (a lane's other scores are at most its
      // second best: when that qualifies too, the record is crowded)
      if (es < kDensePanelSlots) {
        float tn_max = sh.tn[0];
#pragma unroll
        for (int w = 1; w < kMmaWaves; ++w) {
          const float v = sh.tn[w];
          tn_max = (tn_max != tn_max || v != v) ? __builtin_nanf("") : __builtin_fmaxf(tn_max, v);
        }
        const uint32_t s = es;
        const uint32_t kind = sh.slot_kind[s];
        const uint4 h0 = sh.span[s][0];
        const uint4 h1 = sh.span[s][1];
        const uint32_t lo = h0.w;
        const uint32_t cnt = h1.w;
        TileRecord& rec = stage_rec[s];
        if (cnt == 0u) {
          reinterpret_cast<uint4*>(&rec)[0] =
              uint4{__float_as_uint(-__builtin_huge_valf()), 0u, kInvalidToken, lo};
          reinterpret_cast<uint4*>(&rec)[1] =
              uint4{lo, 0u, 0u, __float_as_uint(-__builtin_huge_valf())};
        } else {
          const float* r1 = gl1 + s * kEpiRow;
          const float* r2 = gl2 + s * kEpiRow;
          float G = -__builtin_huge_valf();
          bool fin = true;
#pragma unroll
          for (int u = 0; u < 32; ++u) {
            const float v = r1[u];
            fin &= v == v;
            G = __builtin_fmaxf(G, v);
          }
          const float bs = __builtin_fmaf(tn_max, __builtin_fmaf(a.coef, sh.slot_norm[s], a.coef2),
                                          sh.slot_slack[s]);
          const float L = G - bs;
          const bool finite = fin && bs < 0x1p100f;
          uint32_t members = 0u;  // bit u: lane u's best is a member
          bool crowded = false;
#pragma unroll
          for (int u = 0; u < 32; ++u) {
            members |= (r1[u] + bs >= L) ? (1u << u) : 0u;
            crowded |= r2[u] + bs >= L;
          }
          const uint32_t total = static_cast<uint32_t>(__popc(members));
          const bool ordinary = finite && !crowded && total <= static_cast<uint32_t>(kTileMembers);
          const uint32_t ws[6] = {h0.x, h0.y, h0.z, h1.x, h1.y, h1.z};
          // the tile's lowest allowed token (cnt > 0 bits)
          uint32_t first = kHeadTileTokens;
#pragma unroll
          for (int u = 5; u >= 0; --u) {
            if (ws[u] != 0u) first = u * 32u + static_cast<uint32_t>(__builtin_ctz(ws[u]));
          }
          const uint32_t flags =
              ordinary ? 0u : (finite ? kTileRescoreAll | kTileCrowded : kTileRescoreAll);
          reinterpret_cast<uint4*>(&rec)[0] = uint4{__float_as_uint(L), flags, tok0 + first, lo};
          reinterpret_cast<uint4*>(&rec)[1] =
              uint4{lo, cnt, ordinary ? total : 0u, __float_as_uint(G + bs)};
          if (ordinary) {
            uint32_t k = 0u;
            uint32_t left = members;
            while (left != 0u) {
              const uint32_t u = static_cast<uint32_t>(__builtin_ctz(left));
              left &= left - 1u;
              // half u / 16, column u % 16, block of the half glj
              const uint32_t off = ((u / 16u) * kTBw + glj[s * kEpiRow + u]) * 16u + (u % 16u);
              const float v = r1[u];
              // list position: lo + the allowed tokens below off
              uint32_t pos = tok0 + off;
              if (kind == kSlotList) {
                uint32_t rank = 0u;
#pragma unroll
                for (uint32_t t = 0; t < 6u; ++t) {
                  const uint32_t below = off >= (t + 1u) * 32u ? 0xFFFFFFFFu
                                         : (off > t * 32u ? (1u << (off - t * 32u)) - 1u : 0u);
                  rank += static_cast<uint32_t>(__popc(ws[t] & below));
                }
                pos = lo + rank;
              }
              rec.m[k] = TileMember{tok0 + off, pos, v - bs, v + bs};
              ++k;
            }
          }
        }
      }
      __syncthreads();
      store_records(tile);
    }
  };
  if (copier) {
    copy_tiles();
    return;
  }
  switch (nact) {
    case 4: mfma_tiles.template operator()<4>(); break;
    case 3: mfma_tiles.template operator()<3>(); break;
    case 2: mfma_tiles.template operator()<2>(); break;
    case 1: mfma_tiles.template operator()<1>(); break;
    default: mfma_tiles.template operator()<0>(); break;
  }
}

}  // namespace

hipError_t launch_dense(const DenseArgs& args, hipStream_t stream) {
  if (args.H % 32u != 0 || args.H <= 2u * kKC || args.groups < 8u ||
      args.groups % 8u != 0 || args.z_hi == nullptr || args.spans == nullptr) {
    return hipErrorInvalidValue;
  }
  // every slot needs a panel of this launch: a workgroup past its XCD's
  // panels would return without writing its records and fb_map entries,
  // and the finalize would read stale records
  if (static_cast<uint64_t>(args.fb_m) + args.rows >
      static_cast<uint64_t>(args.groups / 8u) * kDensePanelSlots) {
    return hipErrorInvalidValue;
  }
  const uint32_t lds = dense_lds_bytes();
  hipLaunchKernelGGL(dense_kernel, dim3(args.groups), dim3(kThreads), lds, stream, args);
  return hipGetLastError();
}

}  // namespace mf
