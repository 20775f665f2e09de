// K2c: per-sample weight gradient of a linear layer on gfx950 MFMA.
//
//   dW[b, o, k] = sum_t g[b, t, o] * a[b, t, k]          (b < B, o < D, k < K)
//   dW[b, o, K] = sum_t g[b, t, o]                        (only with has_bias)
//
// Follows materialize_factors for linear layers,
// dattri_llm/gradient/ops/materialize.py:114-116 (torch.bmm(g^T, a) flattened
// to (B, out*in), index o*K + i), with the bias folded as the ones column of
// preprocess.py:436-437 (so the layout is (B, D, K+1)).
//
// Both operands contract over the token axis, which is the slow (row) axis of
// the row-major captures.  Each stage therefore loads 8x8 (bf16/f16) or 4x4
// (fp32) blocks with 16-byte row loads, transposes them in registers and
// stores them into LDS token-contiguous, so the MFMA fragment reads are single
// 16-byte LDS reads.  Consecutive lanes take consecutive token blocks of one
// column block, so the 8 lanes the LDS serves together write one 128-byte row
// (all banks distinct); mapping them to consecutive column blocks instead puts
// their rows 8 apart and folds them onto two bank groups.  A workgroup owns a 128 (o) x 128 (k) output tile of one
// sample; the fp32 accumulators are converted to the output dtype and staged
// through LDS so the tile leaves as coalesced 16-byte row stores.
#include <atomic>

#include "common.h"
#include "split.h"

namespace da {
namespace {

constexpr int kBM = 128;                 // output rows (o) per tile
constexpr int kBN = 128;                 // output cols (k) per tile
constexpr int kRowBytes = 128;           // token bytes per LDS row and stage
constexpr int kLdsRow = kRowBytes + 16;  // padded LDS row
constexpr int kThreads = 256;
constexpr int kGroup = 8;
constexpr int kStageBytes = (kBM + kBN) * kLdsRow;

struct MatArgs {
  const char* a;
  const char* g;
  int64_t batch, tokens, k, d;               // k, d: element widths of a, g
  int64_t a_bstride, a_tstride;              // bytes
  int64_t g_bstride, g_tstride;              // bytes
  char* out;
  int64_t out_bstride, out_rstride;          // elements
  int64_t out_blk;                           // elements between 64-element output blocks
  int64_t tiles_m, tiles_n;                  // per sample
  int acc;                                   // add to the fp32 output instead of overwriting it
  int whole_samples;                         // tile order: an XCD takes whole samples
  float scale;                               // sym: factor on what reaches the output
  int64_t rows_total;                        // sym with token splits: rows of all splits (sample b holds
                                             // rows b*tokens .. ; the last one may be short), else 0
  int64_t tile0, sym_count;                  // sym: triangle tiles tile0 .. tile0 + sym_count - 1
  int compact;                               // sym: tile t of split b lands at out + (b*sym_count + t) * 256^2
  int64_t a_part, g_part;                    // split fp32 rows (split.h): bytes of one part of a row
  split::Gate gate;                          // split fp32 rows: which of the two launches runs
};

// Element offset (from the sample's base) of output (o, k): flat c = o*rstride + k
// stored in 64-element blocks out_blk apart (out_blk == 64: plain row-major).
__device__ __forceinline__ int64_t out_index(const MatArgs& m, int64_t o, int64_t k) {
  const int64_t c = o * m.out_rstride + k;
  return (c >> 6) * m.out_blk + (c & 63);
}

// 16-byte output stores need whole output chunks inside every row.
template <int OT>
bool aligned_out(const MatArgs& m) {
  constexpr int64_t os = Elem<OT>::kBytes;
  return m.k % (16 / os) == 0 && (m.out_rstride * os) % 16 == 0 && (m.out_blk * os) % 16 == 0 &&
         (m.out_bstride * os) % 16 == 0 && ((uintptr_t)m.out & 15) == 0;
}

// Transpose a VEC x VEC block held as VEC rows of one 16-byte chunk each.
template <int DT>
__device__ __forceinline__ void transpose_block(const u32x4 (&in)[Elem<DT>::kVec],
                                                u32x4 (&out)[Elem<DT>::kVec]) {
  if constexpr (DT == DA_F32) {
#pragma unroll
    for (int c = 0; c < 4; ++c) out[c] = u32x4{in[0][c], in[1][c], in[2][c], in[3][c]};
  } else {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int w = c >> 1;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const uint32_t lo = in[2 * p][w], hi = in[2 * p + 1][w];
        out[c][p] = (c & 1) ? ((lo >> 16) | (hi & 0xffff0000u)) : ((lo & 0xffffu) | (hi << 16));
      }
    }
  }
}

template <int DT, int OT>
__global__ __launch_bounds__(kThreads, 2) void materialize_tiles(MatArgs m) {
  if (split::gate_closed(m.gate)) return;
  constexpr int VEC = Elem<DT>::kVec;           // elements per 16-byte chunk
  constexpr int ES = Elem<DT>::kBytes;
  constexpr int TS = kRowBytes / ES;            // tokens per stage
  constexpr int BLK_T = TS / VEC;               // token blocks per stage
  constexpr int BLK_C = kBM / VEC;              // column blocks per operand tile
  constexpr int BLOCKS = BLK_T * BLK_C;         // blocks per operand per stage
  constexpr int PER_THREAD = BLOCKS / (kThreads / 2);
  static_assert(PER_THREAD >= 1 && BLOCKS % (kThreads / 2) == 0, "stage/block mismatch");

  __shared__ __attribute__((aligned(16))) char smem[2 * kStageBytes];

  const int64_t ntiles = (int64_t)gridDim.x;
  const int64_t logical = xcd_remap(blockIdx.x, ntiles);
  const int64_t per_sample = m.tiles_m * m.tiles_n;
  const int64_t b = logical / per_sample;
  const int64_t rem = logical - b * per_sample;
  // swizzle inside the sample: groups of kGroup row tiles sweep the columns
  const int64_t per_group = (int64_t)kGroup * m.tiles_n;
  const int64_t group = rem / per_group;
  const int64_t first = group * kGroup;
  const int64_t gsize = min(m.tiles_m - first, (int64_t)kGroup);
  const int64_t in_group = rem - group * per_group;
  const int64_t tm = first + in_group % gsize;
  const int64_t tn = in_group / gsize;
  const int64_t o0 = tm * kBM, k0 = tn * kBN;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  // This thread stages operand `side` (0: g -> rows o, 1: a -> rows k).
  const int side = tid / (kThreads / 2);
  const int tsub = tid % (kThreads / 2);
  const char* src = side == 0 ? m.g + b * m.g_bstride : m.a + b * m.a_bstride;
  const int64_t tstride = side == 0 ? m.g_tstride : m.a_tstride;
  const int64_t width = side == 0 ? m.d : m.k;
  const int64_t c0 = side == 0 ? o0 : k0;

  u32x4 blk[PER_THREAD][VEC];
  auto gload = [&](int st) {
#pragma unroll
    for (int q = 0; q < PER_THREAD; ++q) {
      const int bi = tsub + q * (kThreads / 2);
      const int bt = bi % BLK_T, bc = bi / BLK_T;
      const int64_t col = c0 + (int64_t)bc * VEC;
      const bool cin = col < width;
#pragma unroll
      for (int r = 0; r < VEC; ++r) {
        const int64_t t = (int64_t)st * TS + bt * VEC + r;
        blk[q][r] = (cin && t < m.tokens) ? ld16(src + t * tstride + col * ES) : u32x4{0, 0, 0, 0};
      }
    }
  };
  auto lstore = [&](int buf) {
    char* base = smem + buf * kStageBytes + (side == 0 ? 0 : kBM * kLdsRow);
#pragma unroll
    for (int q = 0; q < PER_THREAD; ++q) {
      const int bi = tsub + q * (kThreads / 2);
      const int bt = bi % BLK_T, bc = bi / BLK_T;
      u32x4 tr[VEC];
      transpose_block<DT>(blk[q], tr);
#pragma unroll
      for (int c = 0; c < VEC; ++c) st16(base + (bc * VEC + c) * kLdsRow + bt * 16, tr[c]);
    }
  };

  f32x16 acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) acc[x][y] = f32x16{};

  const int nst = (int)((m.tokens + TS - 1) / TS);
  gload(0);
  lstore(0);
  __syncthreads();
  const int frow = lane & 31, fhalf = lane >> 5;
  for (int st = 0; st < nst; ++st) {
    const int buf = st & 1;
    if (st + 1 < nst) gload(st + 1);
    const char* base = smem + buf * kStageBytes;
#pragma unroll
    for (int kg = 0; kg < kRowBytes / 32; ++kg) {
      u32x4 fa[2], fb[2];
#pragma unroll
      for (int x = 0; x < 2; ++x)
        fa[x] = ld16(base + (64 * wm + 32 * x + frow) * kLdsRow + 32 * kg + 16 * fhalf);
#pragma unroll
      for (int y = 0; y < 2; ++y)
        fb[y] = ld16(base + (kBM + 64 * wn + 32 * y + frow) * kLdsRow + 32 * kg + 16 * fhalf);
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) Mfma32<DT>::mma(acc[x][y], fa[x], fb[y]);
    }
    if (st + 1 < nst) lstore(buf ^ 1);
    __syncthreads();
  }

  // Epilogue: each wave stages its 64x64 output block (output dtype) in LDS,
  // then writes whole rows.  The loop above ended with a barrier, so the
  // stage buffers are free.
  constexpr int OS = Elem<OT>::kBytes;
  constexpr int ROWB = 64 * OS;                   // bytes of one staged row
  char* wbuf = smem + wave * (64 * ROWB);
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 32 * x + acc_row(r, lane), col = 32 * y + acc_col(lane);
        Elem<OT>::store(wbuf, (int64_t)row * 64 + col, acc[x][y][r]);
      }
  __syncthreads();
  const int64_t orow0 = o0 + 64 * wm, ocol0 = k0 + 64 * wn;
  char* obase = m.out + (b * m.out_bstride) * OS;
  constexpr int CH = ROWB / 16;                   // 16-byte chunks per row
  constexpr int ROWS_PER_PASS = 64 / CH;
#pragma unroll
  for (int pass = 0; pass < 64 / ROWS_PER_PASS; ++pass) {
    const int row = pass * ROWS_PER_PASS + lane / CH, ch = lane % CH;
    const int64_t orow = orow0 + row;
    const int64_t ocol = ocol0 + (int64_t)ch * (16 / OS);
    if (orow < m.d && ocol < m.k)
      st16(obase + out_index(m, orow, ocol) * OS, ld16(wbuf + row * ROWB + ch * 16));
  }
}

// Large-tile variant for the big layers: a 256 (o) x 256 (k) tile per
// workgroup, one wave per SIMD, each wave a 128 x 128 block (4 x 4 MFMA blocks,
// 256 fp32 accumulators).  Twice the MFMA work per LDS byte of the 128-tile
// kernel and four times the work per stage to hide the next stage's loads.
namespace big {
constexpr int kBM = 256;
constexpr int kBN = 256;
constexpr int kStageBytes = (kBM + kBN) * kLdsRow;  // 73,728 B; two stages fit LDS
}  // namespace big

template <int DT, int OT>
__global__ __launch_bounds__(kThreads, 1) void materialize_tiles_big(MatArgs m) {
  if (split::gate_closed(m.gate)) return;
  constexpr int VEC = Elem<DT>::kVec;
  constexpr int ES = Elem<DT>::kBytes;
  constexpr int TS = kRowBytes / ES;           // tokens per stage
  constexpr int BLK_T = TS / VEC;              // token blocks per stage
  constexpr int BLK_C = big::kBM / VEC;        // column blocks per operand tile
  constexpr int BLOCKS = BLK_T * BLK_C;        // blocks per operand per stage
  constexpr int PER_THREAD = BLOCKS / (kThreads / 2);
  static_assert(PER_THREAD >= 1 && BLOCKS % (kThreads / 2) == 0, "stage/block mismatch");

  extern __shared__ __attribute__((aligned(16))) char smem[];  // 2 * big::kStageBytes

  const int64_t ntiles = (int64_t)gridDim.x;
  const int64_t logical = xcd_remap(blockIdx.x, ntiles);
  const int64_t per_sample = m.tiles_m * m.tiles_n;
  const int64_t b = logical / per_sample;
  const int64_t rem = logical - b * per_sample;
  const int64_t per_group = (int64_t)kGroup * m.tiles_n;
  const int64_t group = rem / per_group;
  const int64_t first = group * kGroup;
  const int64_t gsize = min(m.tiles_m - first, (int64_t)kGroup);
  const int64_t in_group = rem - group * per_group;
  const int64_t tm = first + in_group % gsize;
  const int64_t tn = in_group / gsize;
  const int64_t o0 = tm * big::kBM, k0 = tn * big::kBN;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  const int side = tid / (kThreads / 2);
  const int tsub = tid % (kThreads / 2);
  const char* src = side == 0 ? m.g + b * m.g_bstride : m.a + b * m.a_bstride;
  const int64_t tstride = side == 0 ? m.g_tstride : m.a_tstride;
  const int64_t width = side == 0 ? m.d : m.k;
  const int64_t c0 = side == 0 ? o0 : k0;

  u32x4 blk[PER_THREAD][VEC];
  auto gload = [&](int st) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < PER_THREAD; ++q) {
      const int bi = tsub + q * (kThreads / 2);
      const int bt = bi % BLK_T, bc = bi / BLK_T;
      const int64_t col = c0 + (int64_t)bc * VEC;
      const bool cin = col < width;
#pragma unroll
      for (int r = 0; r < VEC; ++r) {
        const int64_t t = (int64_t)st * TS + bt * VEC + r;
        blk[q][r] = (cin && t < m.tokens) ? ld16(src + t * tstride + col * ES) : u32x4{0, 0, 0, 0};
      }
    }
  };
  auto lstore = [&](int buf) __attribute__((always_inline)) {
    char* base = smem + buf * big::kStageBytes + (side == 0 ? 0 : big::kBM * kLdsRow);
#pragma unroll
    for (int q = 0; q < PER_THREAD; ++q) {
      const int bi = tsub + q * (kThreads / 2);
      const int bt = bi % BLK_T, bc = bi / BLK_T;
      u32x4 tr[VEC];
      transpose_block<DT>(blk[q], tr);
#pragma unroll
      for (int c = 0; c < VEC; ++c) st16(base + (bc * VEC + c) * kLdsRow + bt * 16, tr[c]);
    }
  };

  f32x16 acc[4][4];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) acc[x][y] = f32x16{};

  const int nst = (int)((m.tokens + TS - 1) / TS);
  gload(0);
  lstore(0);
  __syncthreads();
  const int frow = lane & 31, fhalf = lane >> 5;
  for (int st = 0; st < nst; ++st) {
    const int buf = st & 1;
    if (st + 1 < nst) gload(st + 1);
    const char* base = smem + buf * big::kStageBytes;
#pragma unroll
    for (int kg = 0; kg < kRowBytes / 32; ++kg) {
      u32x4 fa[4], fb[4];
#pragma unroll
      for (int x = 0; x < 4; ++x)
        fa[x] = ld16(base + (128 * wm + 32 * x + frow) * kLdsRow + 32 * kg + 16 * fhalf);
#pragma unroll
      for (int y = 0; y < 4; ++y)
        fb[y] = ld16(base + (big::kBM + 128 * wn + 32 * y + frow) * kLdsRow + 32 * kg + 16 * fhalf);
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) Mfma32<DT>::mma(acc[x][y], fa[x], fb[y]);
    }
    if (st + 1 < nst) lstore(buf ^ 1);
    __syncthreads();
  }

  // Epilogue: each wave stages its 128 x 128 block in LDS (output dtype), in
  // passes of kPassRows rows so fp32 fits, and writes whole 16-byte chunks.
  constexpr int OS = Elem<OT>::kBytes;
  constexpr int kPassRows = OS == 4 ? 64 : 128;
  constexpr int ROWB = 128 * OS;
  char* wbuf = smem + wave * (kPassRows * ROWB);
  const int64_t orow0 = o0 + 128 * wm, ocol0 = k0 + 128 * wn;
  char* obase = m.out + (b * m.out_bstride) * OS;
#pragma unroll
  for (int pass = 0; pass < 128 / kPassRows; ++pass) {
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      if ((32 * x) / kPassRows != pass) continue;
#pragma unroll
      for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = 32 * x + acc_row(r, lane) - pass * kPassRows, col = 32 * y + acc_col(lane);
          Elem<OT>::store(wbuf, (int64_t)row * 128 + col, acc[x][y][r]);
        }
    }
    __syncthreads();
    constexpr int CH = ROWB / 16;
    constexpr int RPP = 64 / CH;  // rows per 64-lane pass
    for (int rr = 0; rr < kPassRows; rr += RPP) {
      const int row = rr + lane / CH, ch = lane % CH;
      const int64_t orow = orow0 + pass * kPassRows + row;
      const int64_t ocol = ocol0 + (int64_t)ch * (16 / OS);
      if (orow < m.d && ocol < m.k)
        st16(obase + out_index(m, orow, ocol) * OS, ld16(wbuf + row * ROWB + ch * 16));
    }
    __syncthreads();
  }
}

// Transposing-read variant for 2-byte inputs (bf16 / f16), used for the large
// layers.  Operand tiles go from HBM to LDS untouched, by buffer loads with the
// LDS-direct bit (16 bytes per lane, nothing staged in VGPRs), and the MFMA
// fragments come out of LDS token-contiguous through ds_read_b64_tr_b16: within
// each 16-lane group, lane j addresses 4 consecutive columns of token row
// (r0 + j/4) and lane i receives tokens r0..r0+3 of column i.  Rows past the
// sample's last token and columns past the width read as zero through the
// buffer range check.  The ring holds four 32-token stages, three in flight
// while the fourth is multiplied (a fifth stage, all 160 KB of LDS, measured
// slower).
namespace trk {
constexpr int kBM = 256;
constexpr int kBN = 256;
constexpr int kGroup = 4;                   // row tiles per column sweep (4 beat 8 and 16 on the C4 dW shapes)
constexpr int kTS = 32;                     // tokens per stage
constexpr int kRow = 512;                   // bytes per token row of a 256-column operand tile
constexpr int kOp = kTS * kRow;             // 16 KB per operand per stage
constexpr int kStage = 2 * kOp;             // g tile, then a tile
constexpr int kNBuf = 4;                    // ring of stages: 128 KB
constexpr uint32_t kOob = 0x80000000u;      // offset past every range: the load returns zeros
// 16-byte chunk c of token row r is stored in slot c ^ swz(r).  One transposing
// read touches 8 token rows (r % 4 = 0..3, twice) x 64 bytes; the swizzle puts
// the four rows of each half in different 64-byte quarters of a 256-byte bank
// sweep.
__device__ __forceinline__ int swz(int r) { return (r & 3) << 2; }
}  // namespace trk

typedef short s16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ u32x4 tr_frag(const lds_char* p0, const lds_char* p1) {
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p0);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p1);
  const u32x2 l = __builtin_bit_cast(u32x2, lo), h = __builtin_bit_cast(u32x2, hi);
  return u32x4{l[0], l[1], h[0], h[1]};
}

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// Store 4 consecutive outputs in the output dtype (round to nearest even).
template <int OT>
__device__ __forceinline__ void store_run4(char* p, float a, float b, float c, float d) {
  if constexpr (OT == DA_F32) {
    *(f32x4*)p = f32x4{a, b, c, d};
  } else if constexpr (OT == DA_BF16) {
    *(u32x2*)p = u32x2{__builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2)),
                       __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{c, d}, bf16x2))};
  } else {
    *(u32x2*)p = u32x2{__builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2)),
                       __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{c, d}, f16x2))};
  }
}

// Tile r of a row Gram's triangle (T x T tiles, tm <= tn): groups of four tile
// rows, swept column by column, so the tiles running together on an XCD (32
// consecutive ones) share their operand columns as in the plain order: 12
// column tiles in place of the 33 of a row-by-row order (7000 rows of 14336 and
// 4096 columns: 1471 us of tiles, 1492 row by row).
__device__ __forceinline__ void triangle_tile(int64_t r, int64_t T, int64_t* tm, int64_t* tn) {
  int64_t first = 0, n = 0, head = 0;
  for (;; first += trk::kGroup) {
    n = min(T - first, (int64_t)trk::kGroup);
    head = n * (n + 1) / 2;                        // the group's own triangle
    const int64_t count = head + n * (T - first - n);
    if (r < count) break;
    r -= count;
  }
  if (r < head) {
    int64_t c = 0;
    while ((c + 1) * (c + 2) / 2 <= r) ++c;
    *tm = first + r - c * (c + 1) / 2;
    *tn = first + c;
  } else {
    r -= head;
    *tm = first + r % n;
    *tn = first + n + r / n;
  }
}

// A 256 x 256 tile on two waves per SIMD (8 waves, 512 threads): wave w owns
// output rows 64 (w / 2) .. +64 and columns 128 (w % 2) .. +128 (2 x 4 MFMA
// blocks, 128 fp32 accumulators, so two waves fit one SIMD's registers).
// While one wave of a SIMD waits at a barrier, on a load or on LDS, the other
// keeps the MFMA pipe busy; four waves of 128 x 128 (one per SIMD) ran 7-11%
// slower on the Llama-3-8B block's shapes (1130-1170 against 1230-1260 TFLOP/s;
// a 5-stage ring and row-tile groups of 2 measured slower, groups of 8 the
// same).  Each 16-token slice costs 6 transposing fragment reads per 8 MFMAs;
// the LDS has the headroom.  Wave w loads token rows 4w .. 4w+3 of both operand
// tiles (2 DMA instructions per operand and stage).
namespace tr8 {
constexpr int kWaves = 8;
constexpr int kThreads = kWaves * kWave;
constexpr int kDma = trk::kTS * (trk::kRow / 16) / (kWave * kWaves);  // per operand and stage
static_assert(kDma == 2, "the vmcnt wait assumes 4 DMA instructions per wave and stage");
enum Stores { kAnyOffset, kChunks, kStream };
}  // namespace tr8

// kStores: 16-byte output stores (kStream: non-temporal ones), or (kAnyOffset,
// plain row-major outputs only) rows at any element offset, in 4-byte stores.  kParts == 3: rows of split fp32 values
// (split.h); the six (g part, a part) segments are walked one after the other,
// each over all tokens.  kSym: a row Gram (a == g), the triangle's tiles on or
// above the diagonal; a tile leaves for its mirrored place as well, straight
// from the accumulators (32 lanes hold 32 consecutive rows of a column, a 128-
// byte run of the mirrored row).  The mirror as a pass of its own read and
// wrote that half again, and the division by the row count was a third pass:
// 2 x 83 us and 2 x 142 us beside 1360 us of tiles on four waves (7000 rows of
// 14336 and 4096 columns); with both in the tiles' epilogue 1471 us in all.
template <int DT, int OT, int kStores, int kParts, bool kSym>
__global__ __launch_bounds__(tr8::kThreads, 1) void materialize_tiles_tr8(MatArgs m) {
  static_assert(Elem<DT>::kBytes == 2, "transposing reads are 16-bit");
  if constexpr (kParts == 3) {
    if (split::gate_closed(m.gate)) return;
  }
  __shared__ __attribute__((aligned(1024))) char smem[trk::kNBuf * trk::kStage];
  lds_char* const L = (lds_char*)smem;
  const uint32_t lds0 = (uint32_t)(uintptr_t)L;

  const int64_t ntiles = (int64_t)gridDim.x;
  const int64_t logical = xcd_remap(blockIdx.x, ntiles);
  int64_t b, tm, tn;
  int64_t sym_local = 0;
  if constexpr (kSym) {
    // Sample b (a token split of the rows), then its tiles tile0 + .. of the
    // triangle (tiles_m == tiles_n).
    b = logical / m.sym_count;
    sym_local = logical - b * m.sym_count;
    triangle_tile(m.tile0 + sym_local, m.tiles_n, &tm, &tn);
  } else {
    // When every sample's tile count divides by 8, XCD x takes the x-th
    // eighth of each sample in turn, so all XCDs stream one sample's factors
    // at a time (a working set the MALL keeps); otherwise, and with
    // whole_samples, XCD x takes the x-th eighth of all tiles.  Within an XCD,
    // the tiles running together are consecutive in groups of kGroup row tiles.
    int64_t rem;
    const int64_t per_sample = m.tiles_m * m.tiles_n;
    if (per_sample % kXcds == 0 && !m.whole_samples) {
      const int64_t chunk = per_sample / kXcds;
      const int64_t xcd = blockIdx.x % kXcds, local = blockIdx.x / kXcds;
      b = local / chunk;
      rem = xcd * chunk + local % chunk;
    } else {
      b = logical / per_sample;
      rem = logical - b * per_sample;
    }
    const int64_t per_group = (int64_t)trk::kGroup * m.tiles_n;
    const int64_t group = rem / per_group;
    const int64_t first = group * trk::kGroup;
    const int64_t gsize = min(m.tiles_m - first, (int64_t)trk::kGroup);
    const int64_t in_group = rem - group * per_group;
    tm = first + in_group % gsize;
    tn = in_group / gsize;
  }
  const int64_t o0 = tm * trk::kBM, k0 = tn * trk::kBN;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;  // 64-row quarter of the g tile, 128-column half of the a tile
  const int uwave = __builtin_amdgcn_readfirstlane(wave);

  // Buffer resources over the sample's token rows (the host guarantees
  // (tokens + kTS) * stride < 2^31, so no offset below wraps).  A token
  // split's end at the last real row: the rows past it (the short last split)
  // read as zeros and touch no memory.
  const int64_t tokens = kSym && m.rows_total > 0 ? min(m.tokens, m.rows_total - b * m.tokens) : m.tokens;
  const u32x4 rg = make_rsrc(m.g + b * m.g_bstride, (uint32_t)(tokens * m.g_tstride));
  const u32x4 ra = make_rsrc(m.a + b * m.a_bstride, (uint32_t)(tokens * m.a_tstride));
  const uint32_t gts = (uint32_t)m.g_tstride, ats = (uint32_t)m.a_tstride;
  const int nseg = (int)((tokens + trk::kTS - 1) / trk::kTS);  // stages per segment
  const int nst = kParts == 3 ? split::kSegs * nseg : nseg;

  // DMA: lane l of instruction j takes token row 4w + 2j + l/32, slot l % 32.
  uint32_t goff[tr8::kDma], aoff[tr8::kDma];
#pragma unroll
  for (int j = 0; j < tr8::kDma; ++j) {
    const int r = 4 * wave + 2 * j + (lane >> 5);
    const int c = (lane & 31) ^ trk::swz(r);
    const int64_t gc = o0 + 8 * c, ac = k0 + 8 * c;
    goff[j] = gc < m.d ? (uint32_t)(r * gts + gc * 2) : trk::kOob;
    aoff[j] = ac < m.k ? (uint32_t)(r * ats + ac * 2) : trk::kOob;
  }
  auto dma_one = [&](int side, int st, int j) __attribute__((always_inline)) {
    const bool en = st < nst;
    const uint32_t lbase = lds0 + (uint32_t)((st % trk::kNBuf) * trk::kStage + side * trk::kOp +
                                             (4 * uwave + 2 * j) * trk::kRow);
    uint32_t step;
    if constexpr (kParts == 3) {
      const int seg = split::segment(st, nseg);
      const uint32_t part = ((side == 0 ? split::kPart1 : split::kPart2) >> (2 * seg)) & 3u;
      step = (uint32_t)(st - seg * nseg) * (trk::kTS * (side == 0 ? gts : ats)) +
             part * (uint32_t)(side == 0 ? m.g_part : m.a_part);
    } else {
      step = (uint32_t)st * (trk::kTS * (side == 0 ? gts : ats));
    }
    const uint32_t off = (side == 0 ? goff[j] : aoff[j]) + step;
    dma16(side == 0 ? rg : ra, lbase, en ? off : trk::kOob);
  };
  auto issue = [&](int st) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < tr8::kDma; ++j) dma_one(0, st, j);
#pragma unroll
    for (int j = 0; j < tr8::kDma; ++j) dma_one(1, st, j);
  };

  // Fragment addresses (lanes as ds_read_b64_tr_b16 wants them): 2 g fragments (rows
  // 64 wm + 32 f) and 4 a fragments (columns 128 wn + 32 f).
  const int q = lane >> 4, i16 = lane & 15;
  const int rsw = (i16 >> 2) << 2;
  const int rowoff = (8 * (q >> 1) + (i16 >> 2)) * trk::kRow;
  int gfr[2], afr[4];
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const int cg = (64 * wm + 32 * f) / 8 + 2 * (q & 1) + ((i16 & 3) >> 1);
    gfr[f] = rowoff + ((cg ^ rsw) << 4) + 8 * (i16 & 1);
  }
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    const int ca = (128 * wn + 32 * f) / 8 + 2 * (q & 1) + ((i16 & 3) >> 1);
    afr[f] = trk::kOp + rowoff + ((ca ^ rsw) << 4) + 8 * (i16 & 1);
  }

  f32x16 acc[2][4];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) acc[x][y] = f32x16{};

  u32x4 f0a[2], f0b[4], f1a[2], f1b[4];
  auto read = [&](const lds_char* sb, u32x4 (&fa)[2], u32x4 (&fb)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < 2; ++f) fa[f] = tr_frag(sb + gfr[f], sb + gfr[f] + 4 * trk::kRow);
#pragma unroll
    for (int f = 0; f < 4; ++f) fb[f] = tr_frag(sb + afr[f], sb + afr[f] + 4 * trk::kRow);
  };
  auto mma = [&](const u32x4 (&fa)[2], const u32x4 (&fb)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 4; ++y) Mfma32<DT>::mma(acc[x][y], fb[y], fa[x]);
  };
  // Wait until this wave's loads of the next stage are done (the 4 * (kNBuf -
  // 2) issued after them may still fly) and its LDS reads have returned, then
  // barrier.
  auto stage_sync = [&]() __attribute__((always_inline)) {
    static_assert(trk::kNBuf == 4, "vmcnt below is 4 * (kNBuf - 2)");
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);
    asm volatile("s_barrier" ::: "memory");
  };
  // Half a stage: the 8 MFMAs of one 16-token slice held in (ua, ub), the 12
  // transposing reads of the next slice into (na, nb), and one operand's 2 DMA
  // instructions of a later stage.  Reads are spread 3 per 2 MFMAs, DMA after
  // the 2nd and 6th MFMA.
  auto half = [&](const u32x4 (&ua)[2], const u32x4 (&ub)[4], const lds_char* sb, u32x4 (&na)[2],
                  u32x4 (&nb)[4], int side, int dst) __attribute__((always_inline)) {
    s16x4 t[12];
    auto rd = [&](int i) __attribute__((always_inline)) {
      const int fr = i >> 1;
      const int fo = fr < 2 ? gfr[fr] : afr[fr - 2];
      t[i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)(sb + fo + (i & 1) * 4 * trk::kRow));
    };
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      rd(i);
      if (i & 1) rd(8 + (i >> 1));
      Mfma32<DT>::mma(acc[i >> 2][i & 3], ub[i & 3], ua[i >> 2]);
      if ((i & 3) == 1 && side >= 0) dma_one(side, dst, i >> 2);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      const u32x2 lo = __builtin_bit_cast(u32x2, t[2 * f]), hi = __builtin_bit_cast(u32x2, t[2 * f + 1]);
      (f < 2 ? na[f] : nb[f - 2]) = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  };

#pragma unroll
  for (int s = 0; s < trk::kNBuf - 1; ++s) issue(s);
  stage_sync();
#pragma unroll
  for (int j = 0; j < tr8::kDma; ++j) dma_one(0, trk::kNBuf - 1, j);
  read(L, f0a, f0b);
  for (int st = 0; st + 1 < nst; ++st) {
    half(f0a, f0b, L + (st % trk::kNBuf) * trk::kStage + 16 * trk::kRow, f1a, f1b, 1, st + trk::kNBuf - 1);
    stage_sync();
    half(f1a, f1b, L + ((st + 1) % trk::kNBuf) * trk::kStage, f0a, f0b, 0, st + trk::kNBuf);
  }
  half(f0a, f0b, L + ((nst - 1) % trk::kNBuf) * trk::kStage + 16 * trk::kRow, f1a, f1b, -1, 0);
  mma(f1a, f1b);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // Epilogue, per 32-row group x of this wave's 64 rows (storing the runs of 4
  // straight to HBM would put the 32 rows of one instruction a row stride
  // apart; at 8 KB strides they serialize on one memory channel):
  // lane l of acc[x][y] holds row o = 32x + l%32 and columns 32y + 8q + 4(l/32)
  // + (0..3) in acc[x][y][4q .. 4q+3].  A wave stages RG rows at a time in its
  // own padded LDS rows (16 when 8 waves' 32 fp32 rows would exceed the ring).
  constexpr int OS = Elem<OT>::kBytes;
  constexpr int ROWB = 128 * OS;
  constexpr int LROW = ROWB + 16;
  constexpr int CH = ROWB / 16;
  constexpr int RPI = kWave / CH;
  constexpr int RG = tr8::kWaves * 32 * LROW <= (int)sizeof(smem) ? 32 : 16;
  static_assert(tr8::kWaves * RG * LROW <= (int)sizeof(smem), "epilogue staging exceeds the ring");
  char* wbuf = smem + wave * (RG * LROW);
  const int h = lane >> 5, ol = lane & 31;
  const int64_t ocol0 = k0 + 128 * wn;
  char* obase = m.out + (b * m.out_bstride) * OS;
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int x = 0; x < 2; ++x) {
#pragma unroll
    for (int p = 0; p < 32 / RG; ++p) {
      if (ol / RG == p) {
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4) {
            const f32x16& v = acc[x][y];
            store_run4<OT>(wbuf + (ol % RG) * LROW + (32 * y + 8 * q4 + 4 * h) * OS, v[4 * q4], v[4 * q4 + 1],
                           v[4 * q4 + 2], v[4 * q4 + 3]);
          }
      }
      // Other lanes of the wave read these rows: no barrier is needed (one wave's
      // LDS operations keep their order), but the compiler must not carry a
      // lane's earlier reads across another lane's writes.
      asm volatile("" ::: "memory");
      if constexpr (kStores == tr8::kAnyOffset) {
        for (int row = 0; row < RG; ++row) {
          const int64_t orow = o0 + 64 * wm + 32 * x + p * RG + row;
          if (orow >= m.d) break;
          char* const dst = obase + (orow * m.out_rstride + ocol0) * OS;
          const char* const srow = wbuf + row * LROW;
          const int n = (int)min((int64_t)128, m.k - ocol0);  // live columns (may be <= 0)
          if constexpr (OS == 4) {
#pragma unroll
            for (int e = lane; e < 128; e += kWave)
              if (e < n) *(uint32_t*)(dst + 4 * e) = *(const uint32_t*)(srow + 4 * e);
          } else {
            // pairs at 4-byte addresses: from element 1 on when the row starts off one
            const int odd = (int)(((uintptr_t)dst >> 1) & 1);
            const int e = 2 * lane + odd;
            const uint16_t* const s16 = (const uint16_t*)srow;
            if (e + 1 < n) *(uint32_t*)(dst + 2 * e) = (uint32_t)s16[e] | ((uint32_t)s16[e + 1] << 16);
            else if (e < n) *(uint16_t*)(dst + 2 * e) = s16[e];
            if (odd && lane == 0 && n > 0) *(uint16_t*)dst = s16[0];
          }
        }
        asm volatile("" ::: "memory");
        continue;
      }
#pragma unroll
      for (int rr = 0; rr < RG; rr += RPI) {
        const int row = rr + lane / CH, ch = lane % CH;
        const int64_t orow = o0 + 64 * wm + 32 * x + p * RG + row;
        const int64_t ocol = ocol0 + (int64_t)ch * (16 / OS);
        u32x4 val = ld16(wbuf + row * LROW + ch * 16);
        if (orow < m.d && ocol < m.k) {
          char* dst = obase + out_index(m, orow, ocol) * OS;
          if constexpr (kSym) {
            f32x4 v = __builtin_bit_cast(f32x4, val);
            if (m.compact) {
              dst = m.out + ((b * m.sym_count + sym_local) * (int64_t)(trk::kBM * trk::kBN) +
                             (orow - o0) * trk::kBN + (ocol - k0)) * OS;
            } else {
              if (m.acc) v += __builtin_bit_cast(f32x4, ld16(dst));
              v *= m.scale;
            }
            val = __builtin_bit_cast(u32x4, v);
          }
          if constexpr (kStores == tr8::kStream) __builtin_nontemporal_store(val, (u32x4*)dst);
          else st16(dst, val);
        }
      }
      asm volatile("" ::: "memory");
    }
  }
  if constexpr (kSym) {
    if (m.compact || tm == tn) return;
    float* const out = (float*)m.out;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int64_t i = k0 + 128 * wn + 32 * y + acc_row(e, lane);  // mirrored row: the column
          const int64_t j = o0 + 64 * wm + 32 * x + ol;
          if (i < m.k && j < m.d) {
            float* const p = out + i * m.out_rstride + j;
            *p = (m.acc ? acc[x][y][e] + *p : acc[x][y][e]) * m.scale;
          }
        }
  }
}

// Narrow layers: one side at most 64 wide (LoRA adapters, small heads).  The
// wide-tile kernels pad such a side to their 128 or 256 rows and leave few
// tiles per sample (16 of 256 x 256 for 4096 -> 16), so the GPU idles and the
// bytes, which bound this shape, stream slowly.  Here a workgroup owns the
// whole narrow side (up to 64 columns) against 64 columns of the wide side:
// 64 tiles per sample at width 4096.  The tile's two 64-column operand slices
// go HBM -> LDS by buffer loads with the LDS-direct bit, 32 tokens per stage
// (8 KB), through a ring of four stages, three in flight, one DMA instruction
// per operand, wave and stage.  Wave w multiplies all (up to four) 16-row
// blocks of the narrow side against wide columns 16w .. 16w+15 with
// 16x16x32 MFMAs, fragments read with transposing LDS reads (16-byte chunk c
// of token row r stored at slot c ^ 2(r % 4), so the four rows of a read's
// 16-lane phase use distinct 32-byte bank groups).  The wide operand is read
// once (non-temporal); the narrow one, shared by the sample's tiles, through
// L2, each XCD owning a contiguous run of tiles.
namespace nw {
constexpr int kCols = 64;            // columns per operand and tile
constexpr int kTS = 32;              // tokens per stage
constexpr int kRow = kCols * 2;      // 128 bytes per token row and operand
constexpr int kSide = kTS * kRow;    // 4 KB
constexpr int kStage = 2 * kSide;    // narrow operand, then wide operand
constexpr int kNBuf = 4;             // three stages in flight (eight measured slower)
constexpr uint32_t kOob = 0x80000000u;
__device__ __forceinline__ int swz(int r) { return (r & 3) << 1; }
static_assert(kNBuf == 4, "the vmcnt wait below is 2 * (kNBuf - 2) = 4");
}  // namespace nw

template <int DT, int OT>
__global__ __launch_bounds__(256) void materialize_narrow(MatArgs m, int narrow_is_d) {
  static_assert(Elem<DT>::kBytes == 2, "transposing reads are 16-bit");
  __shared__ __attribute__((aligned(1024))) char smem[nw::kNBuf * nw::kStage];
  lds_char* const L = (lds_char*)smem;
  const uint32_t lds0 = (uint32_t)(uintptr_t)L;
  const int64_t logical = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t b = logical / m.tiles_n, tw = logical - b * m.tiles_n;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int uwave = __builtin_amdgcn_readfirstlane(wave);

  // the narrow operand (width N) and the wide one (width W) of sample b
  const char* xn = narrow_is_d ? m.g + b * m.g_bstride : m.a + b * m.a_bstride;
  const char* xw = narrow_is_d ? m.a + b * m.a_bstride : m.g + b * m.g_bstride;
  const uint32_t tsn = (uint32_t)(narrow_is_d ? m.g_tstride : m.a_tstride);
  const uint32_t tsw = (uint32_t)(narrow_is_d ? m.a_tstride : m.g_tstride);
  const int64_t n_cols = narrow_is_d ? m.d : m.k, w_cols = narrow_is_d ? m.k : m.d;
  const int64_t w0 = tw * nw::kCols;
  const u32x4 rn = uniform4(make_rsrc(xn, (uint32_t)(m.tokens * tsn)));
  const u32x4 rw = uniform4(make_rsrc(xw, (uint32_t)(m.tokens * tsw)));
  const int nst = (int)((m.tokens + nw::kTS - 1) / nw::kTS);

  // DMA: wave w loads token rows 8w .. 8w+7 of both operands; lane l takes
  // row 8w + l/8 and LDS slot l%8, which holds chunk (l%8) ^ swz(row).
  const int r = 8 * wave + (lane >> 3);
  const int c = (lane & 7) ^ nw::swz(r);
  const uint32_t offn = 8 * c < n_cols ? r * tsn + 16u * (uint32_t)c : nw::kOob;
  const uint32_t offw = w0 + 8 * c < w_cols ? r * tsw + (uint32_t)(w0 + 8 * c) * 2u : nw::kOob;
  auto issue = [&](int st) __attribute__((always_inline)) {
    const bool en = st < nst;
    const uint32_t base = lds0 + (uint32_t)((st % nw::kNBuf) * nw::kStage + 8 * uwave * nw::kRow);
    dma16(rn, base, en && offn != nw::kOob ? offn + (uint32_t)st * (nw::kTS * tsn) : nw::kOob);
    dma16_nt(rw, base + nw::kSide, en && offw != nw::kOob ? offw + (uint32_t)st * (nw::kTS * tsw) : nw::kOob);
  };

  // Fragment of the 16 columns c0 .. c0+15 of one operand over the stage's 32
  // tokens: lane l gets tokens 8(l/16) .. +7 of column c0 + l%16 (two
  // transposing reads of 4 tokens; lane j of a 16-lane phase addresses token
  // row t0 + j/4, columns c0 + 4(j%4) .. +3).
  const int g4 = lane >> 4, i16 = lane & 15;
  auto frag = [&](const lds_char* side, int c0) __attribute__((always_inline)) {
    u32x2 h[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int t = 8 * g4 + 4 * k + (i16 >> 2);
      const int col = c0 + 4 * (i16 & 3);
      const lds_char* p = side + t * nw::kRow + (((col >> 3) ^ nw::swz(t)) << 4) + (col & 7) * 2;
      h[k] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                           (__attribute__((address_space(3))) s16x4*)p));
    }
    return u32x4{h[0][0], h[0][1], h[1][0], h[1][1]};
  };

  const int nblk = (int)((n_cols + 15) / 16);  // 16-row blocks of the narrow side (<= 4)
  f32x4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s0 = 0; s0 < nw::kNBuf - 1; ++s0) issue(s0);
  for (int st = 0; st < nst; ++st) {
    // this wave's loads of stage st are done (the two later stages' 4 may fly),
    // its LDS reads of stage st - 1 have returned; then every wave's
    asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);
    asm volatile("s_barrier" ::: "memory");
    issue(st + nw::kNBuf - 1);  // into the slot stage st - 1 used
    const lds_char* sb = L + (st % nw::kNBuf) * nw::kStage;
    const u32x4 fw = frag(sb + nw::kSide, 16 * wave);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j < nblk) Mfma16<DT>::mma(acc[j], frag(sb, 16 * j), fw);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the zero-fill loads past the last stage

  // lane l holds narrow rows 16j + 4(l/16) + e against wide column 16w + l%16
  const int64_t wc = w0 + 16 * wave + i16;
  if (wc >= w_cols) return;
  const int64_t base = b * m.out_bstride;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (j >= nblk) break;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t n = 16 * j + 4 * g4 + e;
      if (n < n_cols) {
        const int64_t o = narrow_is_d ? n : wc, k = narrow_is_d ? wc : n;
        Elem<OT>::store(m.out, base + out_index(m, o, k), acc[j][e]);
      }
    }
  }
}

// Small layers, several per launch.  A 128-wide layer is one 128 x 128 tile per
// sample: 32 workgroups on 256 CUs, a few stages each, then another launch for
// the bias column and the next layer's after that.  Here a workgroup takes a 64
// x 64 tile of one sample of one of the launch's layers (four waves of one 32 x
// 32 MFMA block), so the layers of a block fill the chip together, and tiles
// of the first 64 input columns also sum their staged gradient columns: the
// bias column.  Stages are 128 bytes of tokens per column, transposed in
// registers on their way to LDS as in materialize_tiles.  Thirteen layers of
// a 128-wide decoder, 32 and 8 samples of 64 fp32 tokens: 26 launches of 14.8 us
// and 26 bias launches of 12.9 us before, two launches of 36 us with it.
namespace grp {
constexpr int kT = 64;                         // output rows and columns per tile
constexpr int kMaxLayers = 24;                 // per launch (the argument block stays under 4 KB)
constexpr int kStageBytes = 2 * kT * kLdsRow;  // 18 KB, double buffered
struct Layer {
  const char* a;
  const char* g;
  char* out;
  int64_t tokens, k, d;                                  // elements
  int64_t a_bstride, a_tstride, g_bstride, g_tstride;    // bytes
  int64_t out_bstride, out_rstride, out_blk;             // elements
  int64_t tile0, tiles_m, tiles_n;                       // first tile of the launch; tiles per sample
  int bias, aligned;                                     // aligned: 16-byte output stores
};
struct Args {
  Layer layers[kMaxLayers];
  int n_layers;
  split::Gate gate;
};
static_assert(sizeof(Args) <= 4096, "kernel arguments");
}  // namespace grp

template <int DT, int OT>
__global__ __launch_bounds__(kThreads, 4) void materialize_group(grp::Args ga) {
  constexpr int VEC = Elem<DT>::kVec;
  constexpr int ES = Elem<DT>::kBytes;
  constexpr int OS = Elem<OT>::kBytes;
  constexpr int TS = kRowBytes / ES;               // tokens per stage
  constexpr int BLK_T = TS / VEC;                  // 8 token blocks per stage
  constexpr int BLOCKS = BLK_T * (grp::kT / VEC);  // blocks per operand and stage: 128 (fp32), 64
  static_assert(BLOCKS <= kThreads / 2, "one block per thread");
  __shared__ __attribute__((aligned(16))) char smem[2 * grp::kStageBytes];
  if (split::gate_closed(ga.gate)) return;

  int l = 0;
  while (l + 1 < ga.n_layers && ga.layers[l + 1].tile0 <= (int64_t)blockIdx.x) ++l;
  const grp::Layer& m = ga.layers[l];
  const int64_t rem0 = (int64_t)blockIdx.x - m.tile0, per_sample = m.tiles_m * m.tiles_n;
  const int64_t b = rem0 / per_sample, rem = rem0 - b * per_sample;
  const int64_t tm = rem / m.tiles_n, tn = rem - tm * m.tiles_n;
  const int64_t o0 = tm * grp::kT, k0 = tn * grp::kT;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  // This thread stages one block of operand `side` (0: g -> rows o, 1: a -> rows k).
  const int side = tid / (kThreads / 2), bi = tid % (kThreads / 2);
  const int bt = bi % BLK_T, bc = bi / BLK_T;
  const char* src = side == 0 ? m.g + b * m.g_bstride : m.a + b * m.a_bstride;
  const int64_t tstride = side == 0 ? m.g_tstride : m.a_tstride;
  const int64_t col = (side == 0 ? o0 : k0) + (int64_t)bc * VEC;
  const bool stages = bi < BLOCKS;
  const bool cin = stages && col < (side == 0 ? m.d : m.k);
  u32x4 blk[VEC];
  auto gload = [&](int st) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < VEC; ++r) {
      const int64_t t = (int64_t)st * TS + bt * VEC + r;
      blk[r] = cin && t < m.tokens ? ld16(src + t * tstride + col * ES) : u32x4{0, 0, 0, 0};
    }
  };
  auto lstore = [&](int buf) __attribute__((always_inline)) {
    if (!stages) return;
    char* base = smem + buf * grp::kStageBytes + (side == 0 ? 0 : grp::kT * kLdsRow);
    u32x4 tr[VEC];
    transpose_block<DT>(blk, tr);
#pragma unroll
    for (int c = 0; c < VEC; ++c) st16(base + (bc * VEC + c) * kLdsRow + bt * 16, tr[c]);
  };

  f32x16 acc = {};
  const bool sums = m.bias && tn == 0 && tid < grp::kT;  // this thread sums gradient column o0 + tid
  float bsum = 0.f;
  const int nst = (int)((m.tokens + TS - 1) / TS);
  gload(0);
  lstore(0);
  __syncthreads();
  const int frow = lane & 31, fhalf = lane >> 5;
  for (int st = 0; st < nst; ++st) {
    const int buf = st & 1;
    if (st + 1 < nst) gload(st + 1);
    const char* base = smem + buf * grp::kStageBytes;
#pragma unroll
    for (int kg = 0; kg < kRowBytes / 32; ++kg) {
      const u32x4 fa = ld16(base + (32 * wm + frow) * kLdsRow + 32 * kg + 16 * fhalf);
      const u32x4 fb = ld16(base + (grp::kT + 32 * wn + frow) * kLdsRow + 32 * kg + 16 * fhalf);
      Mfma32<DT>::mma(acc, fa, fb);
    }
    if (sums) {
#pragma unroll
      for (int c = 0; c < kRowBytes / 16; ++c) {
        float v[VEC];
        unpack16<DT>(ld16(base + tid * kLdsRow + 16 * c), v);
#pragma unroll
        for (int e = 0; e < VEC; ++e) bsum += v[e];
      }
    }
    if (st + 1 < nst) lstore(buf ^ 1);
    __syncthreads();
  }

  // The tile through LDS (output dtype), then whole rows.
  static_assert(grp::kT * grp::kT * 4 <= 2 * grp::kStageBytes, "the output tile fits the stages");
#pragma unroll
  for (int r = 0; r < 16; ++r)
    Elem<OT>::store(smem, (int64_t)(32 * wm + acc_row(r, lane)) * grp::kT + 32 * wn + acc_col(lane), acc[r]);
  __syncthreads();
  char* obase = m.out + b * m.out_bstride * OS;
  auto at = [&](int64_t o, int64_t k) __attribute__((always_inline)) {
    const int64_t c = o * m.out_rstride + k;
    return obase + ((c >> 6) * m.out_blk + (c & 63)) * OS;
  };
  if (m.aligned) {
    constexpr int CH = grp::kT * OS / 16;  // 16-byte chunks per row
#pragma unroll
    for (int x = tid; x < grp::kT * CH; x += kThreads) {
      const int row = x / CH, ch = x % CH;
      const int64_t o = o0 + row, k = k0 + (int64_t)ch * (16 / OS);
      if (o < m.d && k < m.k) st16(at(o, k), ld16(smem + (row * CH + ch) * 16));
    }
  } else {
    for (int x = tid; x < grp::kT * grp::kT; x += kThreads) {
      const int64_t o = o0 + x / grp::kT, k = k0 + x % grp::kT;
      if (o < m.d && k < m.k) {
        if constexpr (OS == 4) *(uint32_t*)at(o, k) = ((const uint32_t*)smem)[x];
        else *(uint16_t*)at(o, k) = ((const uint16_t*)smem)[x];
      }
    }
  }
  if (sums && o0 + tid < m.d) Elem<OT>::store(at(o0 + tid, m.k), 0, bsum);
}

// Launches the layers, kMaxLayers at a time.  One layer of `m` as the group sees it:
template <int OT>
grp::Layer group_layer(const MatArgs& m, int has_bias) {
  grp::Layer L;
  L.a = m.a;
  L.g = m.g;
  L.out = m.out;
  L.tokens = m.tokens;
  L.k = m.k;
  L.d = m.d;
  L.a_bstride = m.a_bstride;
  L.a_tstride = m.a_tstride;
  L.g_bstride = m.g_bstride;
  L.g_tstride = m.g_tstride;
  L.out_bstride = m.out_bstride;
  L.out_rstride = m.out_rstride;
  L.out_blk = m.out_blk;
  L.tile0 = 0;
  L.tiles_m = (m.d + grp::kT - 1) / grp::kT;
  L.tiles_n = (m.k + grp::kT - 1) / grp::kT;
  L.bias = has_bias;
  L.aligned = aligned_out<OT>(m);
  return L;
}

template <int DT, int OT>
int launch_group(const MatArgs* mats, const int* bias, int n, hipStream_t st) {
  for (int i0 = 0; i0 < n; i0 += grp::kMaxLayers) {
    grp::Args ga;
    ga.n_layers = 0;
    ga.gate = mats[i0].gate;  // one layer at a time when it is set
    int64_t tiles = 0;
    for (int i = i0; i < n && i < i0 + grp::kMaxLayers; ++i) {
      grp::Layer& L = ga.layers[ga.n_layers++] = group_layer<OT>(mats[i], bias[i]);
      L.tile0 = tiles;
      tiles += mats[i].batch * L.tiles_m * L.tiles_n;
    }
    if (tiles > 0x7fffffffLL) return set_error(DA_ERR_INVALID, "da_materialize_linear: too many tiles");
    if (tiles > 0) materialize_group<DT, OT><<<(unsigned)tiles, kThreads, 0, st>>>(ga);
    const int rc = check_launch("da_materialize_linear(group)");
    if (rc) return rc;
  }
  return DA_OK;
}

// Row Gram with token splits: for the triangle tiles tile0 .. tile0 + count - 1
// (triangle_tile's order, T tiles per side), out = (out +) the sum over splits s, in
// order, of the compact partial tiles ws[s][t] (256 x 256 fp32 each), times
// scale, to its place and (through LDS) the mirrored one.  Block (t, y): the 64 x
// 64 outputs y of tile t, four float4 per thread.
__global__ __launch_bounds__(256) void sum_split_tiles(const float* __restrict__ ws, int splits, int64_t count,
                                                       int64_t tile0, int64_t T, int64_t n, float* __restrict__ out,
                                                       int64_t ld, int acc, float scale) {
  __shared__ float tr[64][65];
  const int64_t t = blockIdx.x;
  int64_t tm, tn;
  triangle_tile(tile0 + t, T, &tm, &tn);
  const int r0 = 64 * (int)(blockIdx.y >> 2), c0 = 64 * (int)(blockIdx.y & 3);
  const int64_t i0 = tm * trk::kBM + r0, j0 = tn * trk::kBN + c0;
  const int64_t tile = (int64_t)trk::kBM * trk::kBN;
  // the block's partials lie inside the workspace's whole tiles, past n too
  f32x4 v[4] = {};
  const float* src = ws + t * tile + (int64_t)(r0 + (threadIdx.x >> 4)) * trk::kBN + c0 + 4 * (threadIdx.x & 15);
#pragma unroll 4
  for (int s = 0; s < splits; ++s, src += count * tile)
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] += *(const f32x4*)(src + 16 * k * trk::kBN);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int x = threadIdx.x + 256 * k, row = x >> 4, c4 = 4 * (x & 15);
    const int64_t i = i0 + row, j = j0 + c4;
    if (i < n && j < n) {  // n is a multiple of 8: the float4 lies inside
      float* dst = out + i * ld + j;
      if (acc) v[k] += *(const f32x4*)dst;
      v[k] *= scale;
      *(f32x4*)dst = v[k];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) tr[row][c4 + e] = v[k][e];
  }
  if (tm == tn) return;  // uniform
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int x = threadIdx.x + 256 * k, row = x >> 4, c4 = 4 * (x & 15);
    const int64_t i = j0 + row, j = i0 + c4;  // mirrored row and first column
    if (i < n && j < n)
      *(f32x4*)(out + i * ld + j) = f32x4{tr[c4][row], tr[c4 + 1][row], tr[c4 + 2][row], tr[c4 + 3][row]};
  }
}

// Gradient-free rows: out[r] = 1 when some entry of row r compares unequal to
// zero, by its magnitude bits (-0.0 is zero; NaN, inf and subnormals are not),
// one workgroup per row reading it once in 16-byte chunks.
template <int ES>
__global__ __launch_bounds__(256) void nonzero_rows_kernel(const char* __restrict__ x, int64_t chunks,
                                                           int64_t stride_b, uint8_t* __restrict__ out) {
  const int64_t r = blockIdx.x;
  const u32x4* p = (const u32x4*)(x + r * stride_b);
  constexpr uint32_t kMag = ES == 4 ? 0x7fffffffu : 0x7fff7fffu;  // both halves of a 16-bit pair
  uint32_t any = 0;
  for (int64_t c = threadIdx.x; c < chunks; c += 256) {
    const u32x4 v = __builtin_nontemporal_load(p + c);
    any |= (v[0] & kMag) | (v[1] & kMag) | (v[2] & kMag) | (v[3] & kMag);
  }
  const int nz = __syncthreads_or(any != 0u);
  if (threadIdx.x == 0) out[r] = nz ? 1 : 0;
}

// Bias column dW[b, o, K] = sum_t g[b, t, o] beside the large-tile kernels: a
// workgroup takes 8 chunks of 16 bytes of one sample's gradient columns; its 32
// thread groups stride the tokens and their sums are added in order.  (One
// thread per column, walking all tokens: 119 us for 8 x 509 tokens of 4096 fp32
// columns, 8 us like this.)
template <int DT, int OT>
__global__ __launch_bounds__(256) void bias_column(const char* g, int64_t tokens, int64_t d, int64_t g_bstride,
                                                   int64_t g_tstride, char* out, int64_t out_bstride,
                                                   int64_t out_rstride, int64_t out_blk, int64_t kcol) {
  constexpr int VEC = Elem<DT>::kVec;
  __shared__ float red[32][8 * VEC + 1];
  const int c = threadIdx.x & 7, t0 = threadIdx.x >> 3;
  const int64_t b = blockIdx.y, col = ((int64_t)blockIdx.x * 8 + c) * VEC;
  const char* src = g + b * g_bstride + col * Elem<DT>::kBytes;
  float sum[VEC] = {};
  if (col < d) {
#pragma unroll 4
    for (int64_t t = t0; t < tokens; t += 32) {
      float v[VEC];
      unpack16<DT>(ld16(src + t * g_tstride), v);
#pragma unroll
      for (int e = 0; e < VEC; ++e) sum[e] += v[e];
    }
  }
#pragma unroll
  for (int e = 0; e < VEC; ++e) red[t0][c * VEC + e] = sum[e];
  __syncthreads();
  const int64_t o = (int64_t)blockIdx.x * 8 * VEC + threadIdx.x;
  if (threadIdx.x >= 8 * VEC || o >= d) return;
  float s = 0.f;
  for (int r = 0; r < 32; ++r) s += red[r][threadIdx.x];
  const int64_t f = o * out_rstride + kcol;
  Elem<OT>::store(out, b * out_bstride + (f >> 6) * out_blk + (f & 63), s);
}

// Whether one layer runs on the 64 x 64 tiles of the grouped kernel.  fp32: a
// round of 256 x 256 tiles on the 256 CUs takes about 147 us at 512 tokens, as
// long as 3500 64 x 64 tiles do, so layers that leave the large tiles' last
// round thinly filled go to the small ones (8 x 512 tokens of 1024 x 1024, half a
// round: 93 against 143 us; 2000 tokens of one sample, 16 tiles: 62 against 525;
// 4 x 512 of 2048 x 2048, one whole round: 169 against 147); a side under 256
// leaves the 128 x 128 tiles, two to a CU, which take over from one round on (35
// x 176 tokens of 11840 x 128, 3255 tiles: 212 against 233 us; 5 x 1375 of 64 x
// 128: 106 against 38).  2-byte rows: the transposing-read kernel is several
// times as fast, so only small short layers go to the small tiles (32 x 64
// tokens of 128 x 128: 4.7 against 6.4 us), and with a bias column, whose launch
// of its own they spare, up to 1300 tiles (2 x 512 of 1024 x 1024: 16 against 27
// us; 27 x 205 of 576 x 1152, 4374 tiles: 58 against 46).  Rows off a 16-byte
// boundary have no other kernel where the transposing-read one cannot go.
bool prefer_group(const MatArgs& m, int has_bias, bool aligned, bool tr, int64_t es) {
  const int64_t small = m.batch * ((m.d + grp::kT - 1) / grp::kT) * ((m.k + grp::kT - 1) / grp::kT);
  const int64_t large = m.batch * ((m.d + big::kBM - 1) / big::kBM) * ((m.k + big::kBN - 1) / big::kBN);
  if (!aligned && !tr) return true;
  if (es == 4) {
    if (m.d < big::kBM || m.k < big::kBN) return m.batch * m.tiles_m * m.tiles_n < 512;
    return small < 3500 * ((large + 255) / 256);
  }
  return has_bias ? small <= 1300 : small <= 256 && m.tokens <= 256;
}

// The transposing-read kernel's tiles over `m`'s rows.
template <int DT, int OT, int kParts>
int launch_tr8(const MatArgs& m, bool aligned, hipStream_t st) {
  MatArgs mt = m;
  mt.tiles_m = (m.d + trk::kBM - 1) / trk::kBM;
  mt.tiles_n = (m.k + trk::kBN - 1) / trk::kBN;
  // Small layers: an eighth of a sample is one or a few tiles with no operand in
  // common, so an XCD's 32 tiles would stream 8 to 32 samples' rows; whole samples
  // share theirs (128 samples of 1024 x 1024, 16 tiles: 207 -> 165 us at 512
  // tokens, 85 -> 83 at 128; 8 tiles: 109 -> 85; 24: 266 -> 234).  With few tokens
  // the rows hardly count and the outputs of one sample at a time stream better
  // (32 tokens: 54 against 60 us; 64 tiles at 32 tokens 51 against 59).
  const int64_t per_sample = mt.tiles_m * mt.tiles_n;
  mt.whole_samples = per_sample <= 8 || (per_sample < 64 && m.tokens >= 128);
  // Outputs written past the caches leave them to the operands, and what reads
  // the dense rows next finds no write-back in its way.  dW and its score against
  // 8 dense rows: 4 x 1024 tokens of 4096 x 14336 689 -> 614 us, 1 x 1024 324 -> 266,
  // 32 x 512 of 2048 x 2048 238 -> 204, 4 x 512 46 -> 44, 16 x 512 of 1024 x 1024 38 ->
  // 36; a 4096-wide block against 16 dense rows 3143 -> 2867.  With few tokens a
  // launch is mostly output, and the caches take the bursts: 48 x 128 tokens of
  // 4096 x 4096 469 against 481 us, 8 x 128 72 against 82, 16 x 64 of 2048 x 2048 31.6
  // against 35.6.
  const bool stream = kParts == 1 && m.tokens >= 512;
  const int64_t nt = m.batch * per_sample;
  if (nt > 0x7fffffffLL) return set_error(DA_ERR_INVALID, "da_materialize_linear: too many tiles");
  if (aligned && stream)
    materialize_tiles_tr8<DT, OT, kParts == 1 ? tr8::kStream : tr8::kChunks, kParts, false>
        <<<(unsigned)nt, tr8::kThreads, 0, st>>>(mt);
  else if (aligned)
    materialize_tiles_tr8<DT, OT, tr8::kChunks, kParts, false><<<(unsigned)nt, tr8::kThreads, 0, st>>>(mt);
  else
    materialize_tiles_tr8<DT, OT, tr8::kAnyOffset, kParts, false><<<(unsigned)nt, tr8::kThreads, 0, st>>>(mt);
  return check_launch("da_materialize_linear(transposing reads)");
}

template <int DT, int OT>
int launch_bias(const MatArgs& m, hipStream_t st) {
  constexpr int64_t cols = 8 * Elem<DT>::kVec;
  dim3 grid((unsigned)((m.d + cols - 1) / cols), (unsigned)m.batch);
  bias_column<DT, OT><<<grid, 256, 0, st>>>(m.g, m.tokens, m.d, m.g_bstride, m.g_tstride, m.out, m.out_bstride,
                                            m.out_rstride, m.out_blk, m.k);
  return check_launch("da_materialize_linear(bias)");
}

// Everything but the split form.
template <int DT, int OT>
int launch(const MatArgs& m, int has_bias, hipStream_t st) {
  const int64_t ntiles = m.batch * m.tiles_m * m.tiles_n;
  if (ntiles > 0x7fffffffLL) return set_error(DA_ERR_INVALID, "da_materialize_linear: too many tiles");
  const bool aligned = aligned_out<OT>(m);
  const bool wide = m.d >= big::kBM && m.k >= big::kBN && m.k % 8 == 0;
  // The transposing-read and narrow kernels address a sample's rows with
  // 32-bit buffer offsets and need disjoint rows (a zero token stride would
  // read as empty).
  const int64_t max_ts = m.g_tstride > m.a_tstride ? m.g_tstride : m.a_tstride;
  const bool fits = Elem<DT>::kBytes == 2 && (m.tokens + trk::kTS) * max_ts < (1LL << 31) &&
                    m.g_tstride >= m.d * 2 && m.a_tstride >= m.k * 2;
  const bool use_tr = fits && wide && (aligned || m.out_blk == 64);
  const bool use_narrow = fits && (m.d <= nw::kCols || m.k <= nw::kCols);
  if (!use_narrow && prefer_group(m, has_bias, aligned, use_tr, Elem<DT>::kBytes))
    return launch_group<DT, OT>(&m, &has_bias, 1, st);
  int rc = DA_OK;
  if (use_narrow) {
    MatArgs mn = m;
    const int narrow_is_d = m.d <= nw::kCols ? 1 : 0;
    mn.tiles_m = 1;
    mn.tiles_n = ((narrow_is_d ? m.k : m.d) + nw::kCols - 1) / nw::kCols;
    const int64_t nt = m.batch * mn.tiles_n;
    if (nt > 0x7fffffffLL) return set_error(DA_ERR_INVALID, "da_materialize_linear: too many tiles");
    if constexpr (Elem<DT>::kBytes == 2) materialize_narrow<DT, OT><<<(unsigned)nt, 256, 0, st>>>(mn, narrow_is_d);
    rc = check_launch("da_materialize_linear(narrow)");
  } else if (use_tr) {
    if constexpr (Elem<DT>::kBytes == 2) rc = launch_tr8<DT, OT, 1>(m, aligned, st);
  } else if (aligned && wide) {
    MatArgs mb = m;
    mb.tiles_m = (m.d + big::kBM - 1) / big::kBM;
    mb.tiles_n = (m.k + big::kBN - 1) / big::kBN;
    const int64_t nb = m.batch * mb.tiles_m * mb.tiles_n;
    const size_t lds = 2 * (size_t)big::kStageBytes;
    // Idempotent, so racing first calls are harmless; per template instance.
    static std::atomic<bool> attr_set{false};
    if (!attr_set.load(std::memory_order_relaxed)) {
      if (hipFuncSetAttribute((const void*)materialize_tiles_big<DT, OT>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return set_error(DA_ERR_HIP, "da_materialize_linear: hipFuncSetAttribute failed");
      attr_set.store(true, std::memory_order_relaxed);
    }
    materialize_tiles_big<DT, OT><<<(unsigned)nb, kThreads, lds, st>>>(mb);
    rc = check_launch("da_materialize_linear(big tiles)");
  } else if (ntiles > 0) {
    materialize_tiles<DT, OT><<<(unsigned)ntiles, kThreads, 0, st>>>(m);
    rc = check_launch("da_materialize_linear(tiles)");
  }
  return rc || !has_bias ? rc : launch_bias<DT, OT>(m, st);
}

// Bytes of the split copies of one fp32 layer, 0 when it stays on fp32 rows: a
// 256 x 256 tile's 32-token stage takes about 0.86 us on the bf16 pipe and is
// run six times, 12 us go to a tile's fill and output (18 for rows off a 16-byte
// boundary), the pre-pass moves 10 bytes per value at about 5 TB/s; the fp32
// kernels' times are prefer_group's and, for a 64 x 64 tile's output, 3.5 to 3.8
// ns, or 5.8 for unaligned rows that no cache takes.  With few tokens the outputs
// are what counts: 32 x 64 tokens of 2048 x 2048 with a bias 395 us on the 64 x 64
// tiles and 262 split, 16 x 64 of 4096 x 4096 739 and 438, 64 x 16 of 1024 x 1024
// 135 and 94; 16 x 64 of 4096 x 4096 without one 505 on the large fp32 tiles and
// 386; but 64 x 64 of 512 x 512 with a bias 45 and 51, 128 x 128 122 and 128.
size_t split_bytes(const MatArgs& m, bool aligned) {
  if (m.d < trk::kBM || m.k < trk::kBN || (!aligned && m.out_blk != 64)) return 0;
  const int64_t rows = m.batch * m.tokens;
  const int64_t ts = split::row_bytes(m.d > m.k ? m.d : m.k);
  if ((m.tokens + trk::kTS) * ts >= (1LL << 31)) return 0;
  const size_t bytes = 256 + split::Builder::bytes(rows, m.k) + split::Builder::bytes(rows, m.d);
  if (bytes > split::kMaxBytes) return 0;
  int64_t slots = 0;
  if (device_cu_count(&slots) != DA_OK) return 0;
  const int64_t large = m.batch * ((m.d + trk::kBM - 1) / trk::kBM) * ((m.k + trk::kBN - 1) / trk::kBN);
  const int64_t small = m.batch * ((m.d + grp::kT - 1) / grp::kT) * ((m.k + grp::kT - 1) / grp::kT);
  const double rounds = (double)((large + slots - 1) / slots), tokens = (double)m.tokens;
  const double big_us = aligned ? rounds * (147.0 * tokens / 512.0 + 12.0) : 1e30;
  const bool cached = m.batch * m.d * m.k * 4 < (192LL << 20);
  const double group_us = (double)small * (0.0412 * tokens / 512.0 + (aligned ? 0.0035 : cached ? 0.0038 : 0.0058)) + 8.0;
  const double split_us = rounds * (0.86 * split::kSegs * (double)((m.tokens + trk::kTS - 1) / trk::kTS) +
                                    (aligned ? 12.0 : 18.0)) +
                          (double)rows * (double)(m.k + m.d) * 10.0 / 5e6 + 10.0;
  return split_us < 0.95 * (big_us < group_us ? big_us : group_us) ? bytes : 0;
}

// An fp32 layer on the bf16 pipe, the fp32 kernels behind it for what split
// rows cannot hold.
template <int OT>
int launch_split(const MatArgs& m, int has_bias, void* workspace, hipStream_t st) {
  split::Builder b((char*)workspace, st);
  MatArgs ms = m;
  ms.a = b.add(m.a, m.batch, m.tokens, m.a_bstride, m.a_tstride, m.k);
  ms.g = b.add(m.g, m.batch, m.tokens, m.g_bstride, m.g_tstride, m.d);
  ms.a_tstride = split::row_bytes(m.k);
  ms.g_tstride = split::row_bytes(m.d);
  ms.a_bstride = m.tokens * ms.a_tstride;
  ms.g_bstride = m.tokens * ms.g_tstride;
  ms.a_part = split::part_elems(m.k) * 2;
  ms.g_part = split::part_elems(m.d) * 2;
  int rc = b.flush();
  if (rc) return rc;
  ms.gate = split::Gate{b.flag(), 0};
  rc = launch_tr8<DA_BF16, OT, 3>(ms, aligned_out<OT>(m), st);
  if (rc) return rc;
  MatArgs mf = m;
  mf.gate = split::Gate{b.flag(), 1};
  rc = launch<DA_F32, OT>(mf, 0, st);
  return rc || !has_bias ? rc : launch_bias<DA_F32, OT>(m, st);
}

}  // namespace
}  // namespace da

namespace da {
namespace {

// The checks of one layer and its kernel arguments; *empty: nothing to compute.
int mat_args(const char* who, const void* a, const void* g, int dtype, int64_t batch, int64_t tokens, int64_t K,
             int64_t D, int64_t a_bstride, int64_t a_tstride, int64_t g_bstride, int64_t g_tstride, int has_bias,
             void* out, int out_dtype, int64_t out_bstride, int64_t out_rstride, int64_t out_blk, MatArgs* args,
             bool* empty) {
  *empty = false;
  if (!valid_dtype(dtype) || !valid_dtype(out_dtype)) return set_error(DA_ERR_INVALID, "%s: bad dtype", who);
  if (batch < 0 || tokens < 0 || K < 0 || D < 0) return set_error(DA_ERR_INVALID, "%s: negative size", who);
  if (batch == 0 || K == 0 || D == 0) {
    *empty = true;
    return DA_OK;
  }
  const int64_t es = (int64_t)elem_bytes(dtype);
  if ((K * es) % 16 || (D * es) % 16)
    return set_error(DA_ERR_INVALID, "%s: K and D must be multiples of %lld", who, (long long)(16 / es));
  if (!a || !g || !out) return set_error(DA_ERR_INVALID, "%s: NULL pointer", who);
  if (((uintptr_t)a | (uintptr_t)g) & 15)
    return set_error(DA_ERR_INVALID, "%s: inputs must be 16-byte aligned", who);
  if (((a_bstride * es) | (a_tstride * es) | (g_bstride * es) | (g_tstride * es)) % 16)
    return set_error(DA_ERR_INVALID, "%s: strides must be multiples of 16 bytes", who);
  if (out_rstride < K + (has_bias ? 1 : 0)) return set_error(DA_ERR_INVALID, "%s: out row stride too small", who);
  if (out_blk == 0) out_blk = 64;
  if (out_blk < 64) return set_error(DA_ERR_INVALID, "%s: out_blk must be 0 or >= 64", who);
  if (out_blk != 64 && ((out_rstride % 64) || out_bstride < 64))
    return set_error(DA_ERR_INVALID, "%s: a blocked output needs a row stride multiple of 64 and out_bstride >= 64",
                     who);
  if (tokens == 0) return set_error(DA_ERR_INVALID, "%s: tokens must be >= 1", who);
  MatArgs& m = *args;
  m.a = (const char*)a;
  m.g = (const char*)g;
  m.batch = batch;
  m.tokens = tokens;
  m.k = K;
  m.d = D;
  m.a_bstride = a_bstride * es;
  m.a_tstride = a_tstride * es;
  m.g_bstride = g_bstride * es;
  m.g_tstride = g_tstride * es;
  m.out = (char*)out;
  m.out_bstride = out_bstride;
  m.out_rstride = out_rstride;
  m.out_blk = out_blk;
  m.tiles_m = (D + kBM - 1) / kBM;
  m.tiles_n = (K + kBN - 1) / kBN;
  m.scale = 1.f;
  m.whole_samples = 0;
  m.acc = 0;
  m.rows_total = 0;
  m.tile0 = 0;
  m.sym_count = 0;
  m.compact = 0;
  m.a_part = 0;
  m.g_part = 0;
  m.gate = split::Gate{nullptr, 0};
  return DA_OK;
}

}  // namespace
}  // namespace da

#define DA_MAT_DISPATCH(dtype, out_dtype, CALL)            \
  switch (3 * (dtype) + (out_dtype)) {                     \
    case 3 * DA_BF16 + DA_F32: return CALL(DA_BF16, DA_F32);   \
    case 3 * DA_BF16 + DA_BF16: return CALL(DA_BF16, DA_BF16); \
    case 3 * DA_BF16 + DA_F16: return CALL(DA_BF16, DA_F16);   \
    case 3 * DA_F16 + DA_F32: return CALL(DA_F16, DA_F32);     \
    case 3 * DA_F16 + DA_BF16: return CALL(DA_F16, DA_BF16);   \
    case 3 * DA_F16 + DA_F16: return CALL(DA_F16, DA_F16);     \
    case 3 * DA_F32 + DA_F32: return CALL(DA_F32, DA_F32);     \
    case 3 * DA_F32 + DA_BF16: return CALL(DA_F32, DA_BF16);   \
    default: return CALL(DA_F32, DA_F16);                      \
  }

extern "C" int da_materialize_linear(const void* a, const void* g, int dtype, int64_t batch,
                                     int64_t tokens, int64_t K, int64_t D, int64_t a_bstride,
                                     int64_t a_tstride, int64_t g_bstride, int64_t g_tstride,
                                     int has_bias, void* out, int out_dtype, int64_t out_bstride,
                                     int64_t out_rstride, int64_t out_blk, void* stream) {
  return da_materialize_linear_ws(a, g, dtype, batch, tokens, K, D, a_bstride, a_tstride, g_bstride, g_tstride,
                                  has_bias, out, out_dtype, out_bstride, out_rstride, out_blk, nullptr, 0, stream);
}

extern "C" int da_materialize_linear_workspace_for(int dtype, int64_t batch, int64_t tokens, int64_t K, int64_t D,
                                                   int aligned_rows, size_t* bytes) {
  using namespace da;
  if (!bytes) return set_error(DA_ERR_INVALID, "da_materialize_linear_workspace: bytes is NULL");
  if (!valid_dtype(dtype)) return set_error(DA_ERR_INVALID, "da_materialize_linear_workspace: bad dtype");
  if (batch < 0 || tokens < 0 || K < 0 || D < 0)
    return set_error(DA_ERR_INVALID, "da_materialize_linear_workspace: negative size");
  *bytes = 0;
  if (dtype != DA_F32 || batch == 0 || tokens == 0 || K == 0 || D == 0) return DA_OK;
  MatArgs m;
  m.batch = batch;
  m.tokens = tokens;
  m.k = K;
  m.d = D;
  m.out_blk = 64;
  *bytes = split_bytes(m, aligned_rows != 0);
  return DA_OK;
}

extern "C" int da_materialize_linear_workspace(int dtype, int64_t batch, int64_t tokens, int64_t K, int64_t D,
                                               size_t* bytes) {
  const int rc = da_materialize_linear_workspace_for(dtype, batch, tokens, K, D, 1, bytes);
  if (rc) return rc;
  size_t unaligned = 0;
  da_materialize_linear_workspace_for(dtype, batch, tokens, K, D, 0, &unaligned);
  if (unaligned > *bytes) *bytes = unaligned;
  return DA_OK;
}

extern "C" int da_materialize_linear_ws(const void* a, const void* g, int dtype, int64_t batch, int64_t tokens,
                                        int64_t K, int64_t D, int64_t a_bstride, int64_t a_tstride,
                                        int64_t g_bstride, int64_t g_tstride, int has_bias, void* out, int out_dtype,
                                        int64_t out_bstride, int64_t out_rstride, int64_t out_blk, void* workspace,
                                        size_t workspace_bytes, void* stream) {
  using namespace da;
  MatArgs m;
  bool empty;
  const int rc = mat_args("da_materialize_linear", a, g, dtype, batch, tokens, K, D, a_bstride, a_tstride, g_bstride,
                          g_tstride, has_bias, out, out_dtype, out_bstride, out_rstride, out_blk, &m, &empty);
  if (rc || empty) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == DA_F32 && workspace) {
    const bool aligned = out_dtype == DA_F32    ? aligned_out<DA_F32>(m)
                         : out_dtype == DA_BF16 ? aligned_out<DA_BF16>(m)
                                                : aligned_out<DA_F16>(m);
    const size_t need = split_bytes(m, aligned);
    if (need && workspace_bytes >= need && ((uintptr_t)workspace & 15) == 0) {
      switch (out_dtype) {
        case DA_F32: return launch_split<DA_F32>(m, has_bias, workspace, st);
        case DA_BF16: return launch_split<DA_BF16>(m, has_bias, workspace, st);
        default: return launch_split<DA_F16>(m, has_bias, workspace, st);
      }
    }
  }
#define DA_MAT_ONE(DT, OT) launch<DT, OT>(m, has_bias, st)
  DA_MAT_DISPATCH(dtype, out_dtype, DA_MAT_ONE)
#undef DA_MAT_ONE
}

extern "C" int da_materialize_linear_group(const da_mat_layer* layers, int n_layers, int dtype, int out_dtype,
                                           void* stream) {
  using namespace da;
  const char* who = "da_materialize_linear_group";
  if (n_layers < 0 || (n_layers > 0 && !layers)) return set_error(DA_ERR_INVALID, "%s: bad layer list", who);
  if (!valid_dtype(dtype) || !valid_dtype(out_dtype)) return set_error(DA_ERR_INVALID, "%s: bad dtype", who);
  hipStream_t st = (hipStream_t)stream;
  for (int pass = 0; pass < 2; ++pass) {  // every layer is checked before the first launch
    MatArgs mats[grp::kMaxLayers];
    int bias[grp::kMaxLayers];
    int n = 0;
    for (int i = 0; i < n_layers; ++i) {
      const da_mat_layer& L = layers[i];
      bool empty;
      int rc = mat_args(who, L.a, L.g, dtype, L.batch, L.tokens, L.K, L.D, L.a_bstride, L.a_tstride, L.g_bstride,
                        L.g_tstride, L.has_bias, L.out, out_dtype, L.out_bstride, L.out_rstride, L.out_blk, &mats[n],
                        &empty);
      if (rc) return rc;
      bias[n] = L.has_bias ? 1 : 0;
      if (pass == 0) continue;
      if (!empty) ++n;
      if (n == grp::kMaxLayers || (i + 1 == n_layers && n > 0)) {
#define DA_MAT_GROUP(DT, OT) launch_group<DT, OT>(mats, bias, n, st)
        rc = [&]() -> int { DA_MAT_DISPATCH(dtype, out_dtype, DA_MAT_GROUP) }();
#undef DA_MAT_GROUP
        if (rc) return rc;
        n = 0;
      }
    }
  }
  return DA_OK;
}

namespace da {
namespace {

struct GramPlan {
  int64_t head;    // triangle tiles 0 .. head - 1 run over all rows, straight into out
  int splits;      // token splits of the remaining tiles (1: no split launch)
  int64_t chunk;   // rows per split
  size_t ws;       // workspace bytes: splits x (tiles - head) compact 256 x 256 fp32 partials
};

// Token splits of a row Gram.  Every tile runs over all the rows, so a triangle
// whose tile count is not a multiple of the CU count ends in a partly filled
// round (width 4096: 136 tiles in one round; width 14336: 1596 tiles, the
// seventh round a quarter full).  The tiles of the whole rounds (head) run as
// they are; the rest are cut into token splits that run side by side, and a
// second pass sums their partial tiles.  Time model in rows of one tile's
// work: a round over `chunk` rows costs `chunk`; the partials' HBM traffic,
// (S + 1) tiles of 256^2 fp32 per split tile at ~5 TB/s against a tile's ~29 ns
// per row on one CU, costs (S + 1) * tiles * 1.8.
GramPlan gram_plan(int64_t rows, int64_t width, int64_t sb, int64_t slots, size_t ws_limit) {
  const int64_t t = (width + trk::kBM - 1) / trk::kBM, nt = t * (t + 1) / 2;
  GramPlan g{nt, 1, rows, 0};
  const int64_t head = nt > slots ? nt / slots * slots : 0, tail = nt - head;
  if (tail == 0) return g;
  const int64_t lim32 = ((1LL << 31) - (1LL << 20)) / sb - trk::kTS;  // rows one buffer resource can span
  const size_t tile_bytes = (size_t)trk::kBM * trk::kBN * sizeof(float);
  // the cheapest split, kept when it beats one pass by 5%
  const double one_pass = (double)((nt + slots - 1) / slots) * (double)rows;
  double best = 0.95 * one_pass;
  for (int s = 2; s <= 64; ++s) {
    int64_t chunk = (rows + s - 1) / s;
    chunk = (chunk + trk::kTS - 1) / trk::kTS * trk::kTS;
    if (chunk < 8 * trk::kTS || chunk > lim32) continue;
    const int64_t sp = (rows + chunk - 1) / chunk;
    if ((size_t)(sp * tail) * tile_bytes > ws_limit || tail * sp > 0x7fffffffLL) continue;
    const double cost = (double)(head / slots) * (double)rows + (double)((tail * sp + slots - 1) / slots) * (double)chunk +
                        1.8 * (double)(sp + 1) * (double)tail;
    if (cost < best) {
      best = cost;
      g = GramPlan{head, (int)sp, chunk, (size_t)(sp * tail) * tile_bytes};
    }
  }
  return g;
}

}  // namespace
}  // namespace da

// Row Gram out = (out +) x^T x of x (rows, width), fp32 out, or that over a
// divisor: the transposing-read dW kernel with every row as one token and both
// operands x, over the tiles on or above the diagonal, each written to its
// mirrored place too.  Tiles run over all rows straight into out, in chunks of
// rows whose buffer offsets fit 32 bits, each adding to the output (the last one
// divides); with token splits (a workspace holding them), the tiles past the
// whole rounds run per split into compact partial tiles, which
// sum_split_tiles adds in split order.
extern "C" int da_row_gram_workspace(int64_t rows, int64_t width, int dtype, size_t* bytes) {
  using namespace da;
  if (!bytes) return set_error(DA_ERR_INVALID, "da_row_gram_workspace: bytes is NULL");
  if (dtype != DA_BF16 && dtype != DA_F16)
    return set_error(DA_ERR_UNSUPPORTED, "da_row_gram_workspace: bf16 or fp16 rows only");
  if (rows < 0 || width < 0) return set_error(DA_ERR_INVALID, "da_row_gram_workspace: negative size");
  *bytes = 0;
  if (rows == 0 || width == 0) return DA_OK;
  int64_t slots = 0;
  const int rc = device_cu_count(&slots);
  if (rc) return rc;
  *bytes = gram_plan(rows, width, width * 2, slots, (size_t)1 << 33).ws;
  return DA_OK;
}

namespace da {
namespace {

int run_row_gram(const void* x, int dtype, int64_t rows, int64_t width, int64_t x_stride, float* out, int64_t ld_out,
                 int accumulate, float scale, void* workspace, size_t workspace_bytes, hipStream_t st) {
  if (dtype != DA_BF16 && dtype != DA_F16)
    return set_error(DA_ERR_UNSUPPORTED, "da_row_gram: bf16 or fp16 rows only");
  if (rows < 0 || width < 0) return set_error(DA_ERR_INVALID, "da_row_gram: negative size");
  if (width == 0) return DA_OK;
  if (!out || (!x && rows > 0)) return set_error(DA_ERR_INVALID, "da_row_gram: NULL pointer");
  const int64_t es = 2;
  if ((width * es) % 16 || (x_stride * es) % 16 || x_stride < width || ((uintptr_t)x & 15))
    return set_error(DA_ERR_INVALID,
                     "da_row_gram: width and row stride must be multiples of 8 elements (stride >= width), "
                     "rows 16-byte aligned");
  if (ld_out < width || (ld_out * 4) % 16 || ((uintptr_t)out & 15))
    return set_error(DA_ERR_INVALID, "da_row_gram: out row stride must be >= width and a multiple of 4");
  if (workspace && ((uintptr_t)workspace & 15))
    return set_error(DA_ERR_INVALID, "da_row_gram: workspace must be 16-byte aligned");
  if (rows == 0) return accumulate ? DA_OK : zero_f32_2d(out, width, width, ld_out, st);
  const int64_t sb = x_stride * es;
  const int64_t chunk32 = ((1LL << 31) - (1LL << 20)) / sb - trk::kTS;
  if (chunk32 < trk::kTS) return set_error(DA_ERR_INVALID, "da_row_gram: rows too wide for 32-bit offsets");
  int64_t slots = 0;
  int rc = device_cu_count(&slots);
  if (rc) return rc;
  const GramPlan g = gram_plan(rows, width, sb, slots, workspace ? workspace_bytes : 0);
  MatArgs m;
  m.batch = 1;
  m.k = width;
  m.d = width;
  m.a_bstride = 0;
  m.g_bstride = 0;
  m.a_tstride = sb;
  m.g_tstride = sb;
  m.out = (char*)out;
  m.out_bstride = 0;
  m.out_rstride = ld_out;
  m.out_blk = 64;
  m.tiles_m = (width + trk::kBM - 1) / trk::kBM;
  m.tiles_n = (width + trk::kBN - 1) / trk::kBN;
  m.rows_total = 0;
  m.whole_samples = 0;
  const int64_t nt = m.tiles_m * (m.tiles_m + 1) / 2;
  m.tile0 = 0;
  m.sym_count = nt;
  m.compact = 0;
  m.a_part = m.g_part = 0;
  m.gate = split::Gate{nullptr, 0};
  auto launch_tiles = [&](int64_t blocks) {
    if (dtype == DA_BF16)
      materialize_tiles_tr8<DA_BF16, DA_F32, tr8::kChunks, 1, true><<<(unsigned)blocks, tr8::kThreads, 0, st>>>(m);
    else
      materialize_tiles_tr8<DA_F16, DA_F32, tr8::kChunks, 1, true><<<(unsigned)blocks, tr8::kThreads, 0, st>>>(m);
    return check_launch("da_row_gram");
  };
  // head: tiles 0 .. head - 1 over all rows, into out (the whole triangle when
  // there are no splits)
  const int64_t head = g.splits > 1 ? g.head : nt;
  if (head > 0) {
    m.sym_count = head;
    for (int64_t r0 = 0; r0 < rows; r0 += chunk32) {
      m.a = (const char*)x + r0 * sb;
      m.g = m.a;
      m.tokens = rows - r0 < chunk32 ? rows - r0 : chunk32;
      m.acc = accumulate || r0 > 0;
      m.scale = r0 + m.tokens == rows ? scale : 1.f;
      rc = launch_tiles(head);
      if (rc) return rc;
    }
  }
  if (g.splits > 1) {
    // tiles head .. nt - 1: split b = rows b*chunk .. of x, compact partial tiles
    const int64_t tail = nt - head;
    m.a = (const char*)x;
    m.g = m.a;
    m.batch = g.splits;
    m.tokens = g.chunk;
    m.rows_total = rows;
    m.a_bstride = g.chunk * sb;
    m.g_bstride = m.a_bstride;
    m.out = (char*)workspace;
    m.tile0 = head;
    m.sym_count = tail;
    m.compact = 1;
    m.acc = 0;
    rc = launch_tiles(tail * g.splits);
    if (rc) return rc;
    sum_split_tiles<<<dim3((unsigned)tail, 16), 256, 0, st>>>((const float*)workspace, g.splits, tail, head,
                                                              m.tiles_m, width, out, ld_out, accumulate ? 1 : 0,
                                                              scale);
    return check_launch("da_row_gram(sum)");
  }
  return DA_OK;
}

}  // namespace
}  // namespace da

extern "C" int da_row_gram(const void* x, int dtype, int64_t rows, int64_t width, int64_t x_stride, float* out,
                           int64_t ld_out, int accumulate, void* workspace, size_t workspace_bytes,
                           void* stream) {
  return da::run_row_gram(x, dtype, rows, width, x_stride, out, ld_out, accumulate, 1.f, workspace, workspace_bytes,
                          (hipStream_t)stream);
}

extern "C" int da_row_gram_mean(const void* x, int dtype, int64_t rows, int64_t width, int64_t x_stride, float* out,
                                int64_t ld_out, int64_t divisor, void* workspace, size_t workspace_bytes,
                                void* stream) {
  if (divisor <= 0) return da::set_error(DA_ERR_INVALID, "da_row_gram_mean: divisor must be positive");
  return da::run_row_gram(x, dtype, rows, width, x_stride, out, ld_out, 0, 1.f / (float)divisor, workspace,
                          workspace_bytes, (hipStream_t)stream);
}

// out[r] = (x[r, :] != 0).any() for the rows of x (rows, width) with row stride
// x_stride (elements): the gradient-free-row test of the K-FAC factors.
extern "C" int da_nonzero_rows(const void* x, int dtype, int64_t rows, int64_t width, int64_t x_stride,
                               uint8_t* out, void* stream) {
  using namespace da;
  if (!valid_dtype(dtype)) return set_error(DA_ERR_INVALID, "da_nonzero_rows: bad dtype %d", dtype);
  if (rows < 0 || width < 0) return set_error(DA_ERR_INVALID, "da_nonzero_rows: negative size");
  if (rows == 0) return DA_OK;
  if (!x || !out) return set_error(DA_ERR_INVALID, "da_nonzero_rows: NULL pointer");
  const int64_t es = (int64_t)elem_bytes(dtype);
  if ((width * es) % 16 || (x_stride * es) % 16 || x_stride < width || ((uintptr_t)x & 15))
    return set_error(DA_ERR_INVALID,
                     "da_nonzero_rows: rows must be 16-byte aligned, width and stride multiples of 16 bytes");
  if (rows > 0x7fffffffLL) return set_error(DA_ERR_INVALID, "da_nonzero_rows: too many rows");
  hipStream_t st = (hipStream_t)stream;
  const int64_t chunks = width * es / 16;
  if (es == 4)
    nonzero_rows_kernel<4><<<(unsigned)rows, 256, 0, st>>>((const char*)x, chunks, x_stride * es, out);
  else
    nonzero_rows_kernel<2><<<(unsigned)rows, 256, 0, st>>>((const char*)x, chunks, x_stride * es, out);
  return check_launch("da_nonzero_rows");
}
