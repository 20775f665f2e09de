// K1: fused ghost inner product (factorized cross-gram) on gfx950 MFMA.
//
//   out[i, j] = sum_{t < S1, s < S2} (a1[i,t,:] . a2[j,s,:]) * (g1[i,t,:] . g2[j,s,:])
//
// Follows the factorized route of cross_gram, dattri_llm/gradient/ops/dot.py:115-118,
// which forms K_a = A1 A2^T and K_g = G1 G2^T as two (B1*S1) x (B2*S2) matrices in
// HBM and then reduces their Hadamard product over each (S1 x S2) block.
//
// Here the same two products are computed as ONE tiled GEMM pair over the row
// spaces (B1*S1) x (B2*S2): a workgroup owns a tile that lies inside a single
// (i, j) sample pair, runs the activation K-loop into one set of fp32 MFMA
// accumulators and the gradient K-loop into a second set, and reduces
// (K_a + bias) * K_g in registers.  Only one fp32 per tile reaches HBM; a
// second tiny kernel sums the per-tile partials of each pair in a fixed order,
// so results are deterministic.
//
// Tile engines: the 256 x 128 tile on 8 waves (ghost_gram_tiles_v3 and the
// grouped MoE form ghost_grouped_tiles_v3, below) takes dense and grouped
// launches whose rows it can address with 32-bit offsets, and the per-token
// form; the 128 x 128 kernels first in this file take per-sample segmented
// sides and the rest.  fp32 factors run the same engine on split rows where
// that pays (split.h): 48 x 24 samples of 201 x 150 tokens, 768 -> 3072, took
// 2396 us on the fp32 matrix pipe and 1865 us split, pre-pass (80 us) included,
// with less than half the error.  Tile order:
// workgroups are remapped so each XCD owns a contiguous run of tiles, grouped
// a few row tiles wide, so the concurrently running tiles on one XCD share
// their operand row blocks through that XCD's L2.
#include <algorithm>
#include <vector>

#include "common.h"
#include "split.h"

namespace da {
namespace {

constexpr int kBM = 128;           // side-1 rows per tile
constexpr int kBN = 128;           // side-2 rows per tile
constexpr int kRowBytes = 128;     // bytes of K consumed per pipeline stage
constexpr int kLdsRow = kRowBytes + 16;  // padded LDS row (bank spread)
constexpr int kThreads = 256;      // 4 waves, 2 x 2 arrangement of 64 x 64
constexpr int kGroup = 8;          // row tiles per swizzle group
constexpr int kStageBytes = (kBM + kBN) * kLdsRow;

struct SideDev {
  const char* act;
  const char* grad;
  int64_t batch, tokens;
  int64_t act_bstride, act_tstride;    // bytes
  int64_t grad_bstride, grad_tstride;  // bytes
  const int32_t* seg;
  const int32_t* idx;
};

using split::Gate;
using split::gate_closed;

struct GhostArgs {
  SideDev s1, s2;
  int64_t kbytes_a, kbytes_g;  // K * esize, D * esize
  int64_t tiles_r, tiles_c;    // tiles per sample on each side
  int64_t n_r, n_c;            // total row / column tiles (diag: n_c = tiles_c)
  float bias;
  int diag;                    // only the pairs (i, i): sample i of side 1 with sample i of side 2
  float* partial;              // [B1][B2][tiles_r][tiles_c], diag: [B][tiles_r][tiles_c]
  Gate gate;
};

// Sample of side 2 for column tile C of row sample i, and the pair's slot in
// the partials.
__device__ __forceinline__ int64_t pair_col_sample(const GhostArgs& g, int64_t i, int64_t C) {
  return g.diag ? i : C / g.tiles_c;
}
__device__ __forceinline__ int64_t pair_slot(const GhostArgs& g, int64_t i, int64_t j) {
  return g.diag ? i : i * g.s2.batch + j;
}

__device__ __forceinline__ int64_t seg_start(const SideDev& s, int64_t b) {
  return s.seg ? (int64_t)s.seg[b] : 0;
}
__device__ __forceinline__ int64_t seg_len(const SideDev& s, int64_t b) {
  return s.seg ? (int64_t)(s.seg[b + 1] - s.seg[b]) : s.tokens;
}
// Byte offset of row t of sample b (t < length) for a factor with the given strides.
__device__ __forceinline__ int64_t row_off(const SideDev& s, int64_t b, int64_t start, int64_t t,
                                           int64_t bstride, int64_t tstride) {
  if (s.seg) {
    const int64_t r = start + t;
    const int64_t p = s.idx ? (int64_t)s.idx[r] : r;
    return p * tstride;
  }
  return b * bstride + t * tstride;
}

// One K-loop of the tile: acc[x][y] += P1[rows 64wm+32x..] . P2[rows 64wn+32y..]^T,
// operands staged through double-buffered LDS, next stage prefetched to registers.
template <int DT>
__device__ __forceinline__ void gram_tile(char* __restrict__ smem, const char* const (&p1)[4],
                                          const char* const (&p2)[4], int64_t kbytes,
                                          f32x16 (&acc)[2][2], int tid, int lane, int wm, int wn) {
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) acc[x][y] = f32x16{};
  const int lr = tid >> 3, lc = tid & 7;
  const int nk = (int)((kbytes + kRowBytes - 1) / kRowBytes);
  u32x4 r1[4], r2[4];

  auto gload = [&](int kt) {
    const int64_t off = (int64_t)kt * kRowBytes + 16 * lc;
    const bool kin = off < kbytes;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      r1[p] = (p1[p] && kin) ? ld16(p1[p] + off) : u32x4{0, 0, 0, 0};
      r2[p] = (p2[p] && kin) ? ld16(p2[p] + off) : u32x4{0, 0, 0, 0};
    }
  };
  auto lstore = [&](int buf) {
    char* base = smem + buf * kStageBytes;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      st16(base + (lr + 32 * p) * kLdsRow + 16 * lc, r1[p]);
      st16(base + (kBM + lr + 32 * p) * kLdsRow + 16 * lc, r2[p]);
    }
  };

  gload(0);
  lstore(0);
  __syncthreads();
  const int frow = lane & 31, fhalf = lane >> 5;
  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < nk) gload(kt + 1);
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
    if (kt + 1 < nk) lstore(buf ^ 1);
    __syncthreads();
  }
}

template <int DT>
__global__ __launch_bounds__(kThreads, 2) void ghost_gram_tiles(GhostArgs g) {
  __shared__ __attribute__((aligned(16))) char smem[2 * kStageBytes];
  __shared__ float red[kThreads / kWave];

  const int64_t logical = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t per_group = (int64_t)kGroup * g.n_c;
  const int64_t group = logical / per_group;
  const int64_t first_r = group * kGroup;
  const int64_t gsize = min(g.n_r - first_r, (int64_t)kGroup);
  const int64_t in_group = logical - group * per_group;
  const int64_t R = first_r + in_group % gsize;
  const int64_t C = in_group / gsize;
  const int64_t i = R / g.tiles_r, tt = R % g.tiles_r;
  const int64_t j = pair_col_sample(g, i, C), ss = C % g.tiles_c;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  const int64_t len1 = seg_len(g.s1, i), len2 = seg_len(g.s2, j);
  const int64_t t0 = tt * kBM, s0 = ss * kBN;
  float* dst = g.partial + (pair_slot(g, i, j) * g.tiles_r + tt) * g.tiles_c + ss;
  if (t0 >= len1 || s0 >= len2) {  // tile entirely past a segment end: contributes 0
    if (tid == 0) *dst = 0.f;
    return;
  }

  const int lr = tid >> 3;
  const int64_t st1 = seg_start(g.s1, i), st2 = seg_start(g.s2, j);
  const char* a1[4];
  const char* g1[4];
  const char* a2[4];
  const char* g2[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int64_t t = t0 + lr + 32 * p;
    const int64_t s = s0 + lr + 32 * p;
    const bool v1 = t < len1, v2 = s < len2;
    a1[p] = v1 ? g.s1.act + row_off(g.s1, i, st1, t, g.s1.act_bstride, g.s1.act_tstride) : nullptr;
    g1[p] = v1 ? g.s1.grad + row_off(g.s1, i, st1, t, g.s1.grad_bstride, g.s1.grad_tstride) : nullptr;
    a2[p] = v2 ? g.s2.act + row_off(g.s2, j, st2, s, g.s2.act_bstride, g.s2.act_tstride) : nullptr;
    g2[p] = v2 ? g.s2.grad + row_off(g.s2, j, st2, s, g.s2.grad_bstride, g.s2.grad_tstride) : nullptr;
  }

  f32x16 ka[2][2], kg[2][2];
  gram_tile<DT>(smem, a1, a2, g.kbytes_a, ka, tid, lane, wm, wn);
  gram_tile<DT>(smem, g1, g2, g.kbytes_g, kg, tid, lane, wm, wn);

  // Rows past a segment end have zero gradient rows, so K_g is 0 there and the
  // bias term (the implicit ones column) contributes nothing for them.
  float s = 0.f;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) s += (ka[x][y][r] + g.bias) * kg[x][y][r];
  s = wave_sum(s);
  if (lane == 0) red[wave] = s;
  __syncthreads();
  if (tid == 0) *dst = (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ void ghost_gram_reduce(const float* __restrict__ partial, int64_t b1, int64_t b2,
                                  int64_t per_pair, float* __restrict__ out, int64_t ld_out,
                                  int accumulate) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= b1 * b2) return;
  const int64_t i = idx / b2, j = idx - i * b2;
  const float* p = partial + idx * per_pair;
  float s = 0.f;
  for (int64_t q = 0; q < per_pair; ++q) s += p[q];
  float* o = out + i * ld_out + j;
  *o = accumulate ? *o + s : s;
}

// ---------------------------------------------------------------------------
// Grouped (MoE) form: tiles over each expert's packed, sample-sorted rows.
// ---------------------------------------------------------------------------
constexpr int kMaxGroups = 16;  // groups per launch (the table travels as kernel arguments)
constexpr int kPRow = kBN + 1; // padded fp32 row of the parked product tile
constexpr int kTileRows = 4;    // row tiles per group of the 256 x 128 tiles' order

struct GroupDev {
  const char* a1;
  const char* g1;
  const char* a2;
  const char* g2;
  const int32_t* seg1;
  const int32_t* seg2;
  const int32_t* idx1;
  const int32_t* idx2;
  int64_t rows1, rows2;               // packed rows per side (seg[B])
  int64_t a1_ts, g1_ts, a2_ts, g2_ts; // row strides, bytes
  int64_t part_off, part_ld;          // partial region (floats) and its row length
  int64_t kbytes_a, kbytes_g;         // K * esize, D * esize
  int64_t slab_off;                   // partial region of the split tiles' slabs
  int32_t tile0;                      // first whole tile of this group in the launch
  int32_t piece0;                     // first piece of this group behind the whole tiles
  int32_t tiles_r, tiles_c;
  int32_t whole;                      // tiles [0, whole) run whole, the rest in pieces
  int16_t pieces_a, pieces_g;         // pieces of a split tile, by product
  float bias;                         // 1 with an implicit ones column, else 0
};

struct GroupedArgs {
  GroupDev grp[kMaxGroups];
  int n_groups;
  int tile_r, tile_c;  // tile heights on side 1 / side 2
  int whole;           // whole tiles of the launch
  int64_t b1, b2;
  float* partial;
  float* dump;         // the pieces' accumulators
  Gate gate;
};
static_assert(sizeof(GroupedArgs) <= 4000, "grouped kernel arguments must stay under 4 KB");

// Row and column of a group's tile `local`: kRows row tiles at a time.
template <int kRows>
__device__ __forceinline__ void group_tile(const GroupDev& G, int32_t local, int32_t& m, int32_t& n) {
  const int32_t grp = local / (kRows * G.tiles_c), first = grp * kRows;
  const int32_t gsize = min(G.tiles_r - first, kRows), in = local - grp * kRows * G.tiles_c;
  m = first + in % gsize;
  n = in / gsize;
}

// Sample owning packed row p < seg[nb]: the last b with seg[b] <= p, or 0.
// The whole wave searches, 64 samples per step.
__device__ __forceinline__ int32_t sample_of(const int32_t* seg, int64_t nb, int64_t p) {
  const int lane = threadIdx.x & 63;
  int32_t lo = 0, n = (int32_t)nb;
  while (n > 1) {
    const int32_t step = (n + 63) / 64;
    const bool below = lane * step < n && (int64_t)seg[lo + lane * step] <= p;
    const int32_t lanes = (int32_t)__popcll(__ballot(below));  // seg does not decrease: a prefix
    const int32_t k = lanes > 0 ? (lanes - 1) * step : 0;
    lo += k;
    n = min(step, n - k);
  }
  return lo;
}

// Sums a parked block of products P (row stride prow) by sample pair: rows
// [t0, t0 + kRB * waves / 2) ∩ [0, n1) of side 1 against the 128 columns from
// s0, ∩ [0, n2).  First every thread walks kRB rows of one column and leaves
// each sample's sum in the first of its rows there (only that thread touches
// those words); then the columns of each (i, j) bin are added, a wave per bin
// where there are few, else a thread.  Bin (i, j) of row block m and column
// tile n goes to part[(i + m) * ld + j + n]: from one bin of a row of tiles to
// the next i or m grows, so i + m tells them apart.  Called by whole
// workgroups, after a barrier behind the parking.
template <int kRB>
__device__ __forceinline__ void pair_bins(float* P, int prow, int64_t t0, int64_t s0, int64_t n1, int64_t n2,
                                          int64_t m, int64_t n, const GroupDev& G, const GroupedArgs& ga,
                                          float* __restrict__ part) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int waves = blockDim.x / kWave;
  {
    const int c = (wave & 1) * 64 + lane;
    const int top = (wave >> 1) * kRB, end = (int)min((int64_t)(top + kRB), n1 - t0);
    int r = (int)max((int64_t)top, (int64_t)G.seg1[0] - t0);  // rows before the first sample belong to none
    if (r < end) {
      int32_t i = sample_of(G.seg1, ga.b1, t0 + r), base = i;
      int32_t ends = G.seg1[min((int64_t)i + 1 + lane, ga.b1)];  // ends of samples base + lane
      while (true) {
        const int e = min(end, (int)(__builtin_amdgcn_readlane(ends, i - base) - t0));
        const int first = r;
        float v = 0.f;
#pragma unroll 8
        for (; r < e; ++r) v += P[r * prow + c];
        if (r > first) P[first * prow + c] = v;
        if (r >= end) break;
        if (++i - base == kWave) {
          base = i;
          ends = G.seg1[min((int64_t)i + 1 + lane, ga.b1)];
        }
      }
    }
  }
  const int64_t last_r = min(t0 + (int64_t)(waves / 2) * kRB, n1) - 1, last_c = min(s0 + kBN, n2) - 1;
  const int32_t i_lo = sample_of(G.seg1, ga.b1, t0), i_hi = sample_of(G.seg1, ga.b1, last_r);
  const int32_t j_lo = sample_of(G.seg2, ga.b2, s0), j_hi = sample_of(G.seg2, ga.b2, last_c);
  const int32_t nj = j_hi - j_lo + 1, nbins = (i_hi - i_lo + 1) * nj;
  __syncthreads();
  const bool by_wave = nbins <= 8 * waves;
  const int step = by_wave ? waves : (int)blockDim.x, lanes = by_wave ? kWave : 1;
  for (int32_t bin = by_wave ? wave : tid; bin < nbins; bin += step) {
    const int32_t i = i_lo + bin / nj, j = j_lo + bin % nj;
    const int r0 = (int)(max((int64_t)G.seg1[i], t0) - t0), r1 = (int)(min((int64_t)G.seg1[i + 1], last_r + 1) - t0);
    const int c0 = (int)(max((int64_t)G.seg2[j], s0) - s0), c1 = (int)(min((int64_t)G.seg2[j + 1], last_c + 1) - s0);
    if (r1 <= r0 || c1 <= c0) continue;  // an empty sample: it owns no slot
    float v = 0.f;
    for (int r = r0; r < r1; r = (r / kRB + 1) * kRB)
      for (int c = c0 + (by_wave ? lane : 0); c < c1; c += lanes) v += P[r * prow + c];
    if (by_wave) v = wave_sum(v);
    if (!by_wave || lane == 0) part[(i + m) * G.part_ld + j + n] = v;
  }
}

template <int DT>
__global__ __launch_bounds__(kThreads, 2) void ghost_grouped_tiles(GroupedArgs ga) {
  __shared__ __attribute__((aligned(16))) char smem[2 * kStageBytes];
  static_assert(kBM * kPRow * 4 <= 2 * kStageBytes, "product tile must fit the stage buffers");

  const int32_t logical = (int32_t)xcd_remap(blockIdx.x, gridDim.x);
  int e = 0;
  while (e + 1 < ga.n_groups && ga.grp[e + 1].tile0 <= logical) ++e;
  const GroupDev& G = ga.grp[e];
  int32_t m, n;
  group_tile<kGroup>(G, logical - G.tile0, m, n);

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int lr = tid >> 3;
  const int64_t t0 = (int64_t)m * kBM, s0 = (int64_t)n * kBN;
  // Rows at or past seg[B] belong to no sample (and may have no row_index
  // entry): treat them as absent; a tile wholly past them has nothing to do.
  const int64_t n1 = min(G.rows1, (int64_t)G.seg1[ga.b1]), n2 = min(G.rows2, (int64_t)G.seg2[ga.b2]);
  if (t0 >= n1 || s0 >= n2) return;
  const char* a1[4];
  const char* g1[4];
  const char* a2[4];
  const char* g2[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int64_t t = t0 + lr + 32 * p, s = s0 + lr + 32 * p;
    const bool v1 = t < n1, v2 = s < n2;
    const int64_t r1 = v1 ? (G.idx1 ? (int64_t)G.idx1[t] : t) : 0;
    const int64_t r2 = v2 ? (G.idx2 ? (int64_t)G.idx2[s] : s) : 0;
    a1[p] = v1 ? G.a1 + r1 * G.a1_ts : nullptr;
    g1[p] = v1 ? G.g1 + r1 * G.g1_ts : nullptr;
    a2[p] = v2 ? G.a2 + r2 * G.a2_ts : nullptr;
    g2[p] = v2 ? G.g2 + r2 * G.g2_ts : nullptr;
  }

  f32x16 ka[2][2], kg[2][2];
  gram_tile<DT>(smem, a1, a2, G.kbytes_a, ka, tid, lane, wm, wn);
  gram_tile<DT>(smem, g1, g2, G.kbytes_g, kg, tid, lane, wm, wn);

  // Park (K_a + bias) * K_g in LDS (rows past an end are zero rows: K_g = 0).
  float* P = (float*)smem;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 64 * wm + 32 * x + acc_row(r, lane), col = 64 * wn + 32 * y + acc_col(lane);
        P[row * kPRow + col] = (ka[x][y][r] + G.bias) * kg[x][y][r];
      }
  __syncthreads();

  pair_bins<64>(P, kPRow, t0, s0, n1, n2, m, n, G, ga, ga.partial + G.part_off);
}

constexpr int kSlab = 64;                     // rows of a split tile that one workgroup finishes
constexpr int kPieceFloats = 256 * 128;       // accumulators of a piece

// out[i, j] (+)= sum over groups of the pair's slots, tile by tile, and slab by
// slab where the tile ran in pieces.  One wave per pair: its lanes are dealt to
// the groups (a power of two each) and within one to the pair's tiles, and
// added by a fixed butterfly (a thread per pair went through 16 groups' slots
// one by one: 47 us for 256 pairs; 6 us).
__global__ __launch_bounds__(256) void grouped_reduce(GroupedArgs ga, float* __restrict__ out, int64_t ld_out,
                                                      int accumulate) {
  const int64_t idx = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  if (idx >= ga.b1 * ga.b2) return;
  const int lane = threadIdx.x & 63;
  const int64_t i = idx / ga.b2, j = idx - i * ga.b2;
  const bool pieces = !gate_closed(ga.gate);
  int per = kWave;  // lanes per group
  while (per * ga.n_groups > kWave) per >>= 1;
  float v = 0.f;
  const int e = lane / per;
  if (e < ga.n_groups) {
    const GroupDev& G = ga.grp[e];
    const int64_t r0 = G.seg1[i], r1 = min((int64_t)G.seg1[i + 1], G.rows1);
    const int64_t c0 = G.seg2[j], c1 = min((int64_t)G.seg2[j + 1], G.rows2);
    if (r0 >= 0 && c0 >= 0 && r1 > r0 && c1 > c0) {
      const int32_t m0 = (int32_t)(r0 / ga.tile_r), nm = (int32_t)((r1 - 1) / ga.tile_r) - m0 + 1;
      const int32_t n0 = (int32_t)(c0 / ga.tile_c), nn = (int32_t)((c1 - 1) / ga.tile_c) - n0 + 1;
      const bool split = pieces && G.whole < G.tiles_r * G.tiles_c;
      const float* part = ga.partial + G.part_off;
      for (int64_t t = lane % per; t < (int64_t)nm * nn; t += per) {
        const int32_t m = m0 + (int32_t)(t / nn), n = n0 + (int32_t)(t % nn);
        const int32_t first = m / kTileRows * kTileRows;
        if (split && first * G.tiles_c + n * min(G.tiles_r - first, kTileRows) + m - first >= G.whole) {
          const int32_t slabs = ga.tile_r / kSlab, s1 = min((int32_t)((r1 - 1) / kSlab), m * slabs + slabs - 1);
          for (int32_t s = max((int32_t)(r0 / kSlab), m * slabs); s <= s1; ++s)
            v += ga.partial[G.slab_off + (i + s) * G.part_ld + j + n];
        } else {
          v += part[(i + m) * G.part_ld + j + n];
        }
      }
    }
  }
  v = wave_sum(v);
  if (lane == 0) {
    float* o = out + i * ld_out + j;
    *o = accumulate ? *o + v : v;
  }
}

// ---------------------------------------------------------------------------
// 256 x 128 tile engine (the gfx950 path).
//
// Both Gram products of a tile -- K_a over the activation width, then K_g over
// the gradient width -- run as ONE stream of 128-byte K stages (one cache line
// of every operand row) through a ring of three LDS stages (48 KB each, two in
// flight).  Operand rows go HBM -> LDS untouched by buffer loads with the
// LDS-direct bit (16 bytes per lane); rows past a sample's end, and chunks past
// the width, read as zero (offset past the buffer range).  Eight waves, two per
// SIMD, each own a 64 x 64 block of both products (2 x 2 MFMA blocks of
// 32 x 32, 128 accumulators), so one wave of a SIMD keeps the MFMA pipe busy
// while the other waits at a barrier, for a load or on LDS.  As in the dW
// kernel, the loads are issued as inline assembly with explicit vmcnt waits,
// interleaved with the MFMAs (a quarter stage of loads per quarter stage of
// MFMAs), and the last quarter of each stage is multiplied after the barrier
// that opens the next.
// ---------------------------------------------------------------------------
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

namespace v2 {
constexpr int kBM = 256;                 // side-1 rows per tile
constexpr int kBN = 128;                 // side-2 rows per tile
constexpr int kRows = kBM + kBN;         // LDS rows per stage
constexpr int kSB = 128;                 // bytes of K per row and stage: one cache line, four 32-byte slices
constexpr int kStage = kRows * kSB;      // 48 KB
constexpr int kNBuf = 3;                 // ring: two stages in flight
constexpr uint32_t kOob = 0x80000000u;
constexpr int kPRow = kBN + 1;           // parked fp32 product row (grouped epilogue)
constexpr int kRing = kNBuf * kStage;
constexpr int kPark = kBM * kPRow * 4;
constexpr int kSmem = kPark > kRing ? kPark : kRing;
static_assert(kSmem <= 160 * 1024, "LDS");
// 16-byte chunk c of LDS row r sits in slot c ^ (r & 7): the 8 lanes one LDS
// cycle serves (8 consecutive rows, one chunk) read 8 distinct bank groups.
}  // namespace v2

// ---------------------------------------------------------------------------
// The engine's per-wave layout: wave w owns the 64 x 64 block at side-1 rows
// 64 (w / 2) and side-2 rows 64 (w % 2); a 32-byte K slice costs it 4 fragment
// reads per 4 MFMAs.  A wave whose block has no live rows or columns only loads
// (TileSrc8::live); waves w and w + 4 share a SIMD, so up to 128 live rows
// leave every SIMD one wave with work.  42 x 48384 rows of 256 + 4488 fp32
// values, token scores: 1142 -> 618 us; 8 experts' packed rows, a few past whole
// tiles: 1056 -> 1019.  Blocks dealt so that 64 live columns do the same cost
// full tiles 0.7% and gave nothing more.  Each wave issues 6 DMA instructions per stage (wave w
// loads tile rows 48w .. 48w+47).
// ---------------------------------------------------------------------------
namespace v3 {
constexpr int kWaves = 8;
constexpr int kThreads = kWaves * kWave;
constexpr int kDma = v2::kRows * (v2::kSB / 16) / (kWave * kWaves);  // 6 per wave and stage
static_assert(kDma == 6, "the vmcnt wait and the quarter split assume 6 DMA instructions per stage");
// instructions [kLo[q], kLo[q + 1]) of a stage go out in quarter q
__device__ __forceinline__ constexpr int lo(int q) { return q == 0 ? 0 : q == 1 ? 2 : q == 2 ? 3 : q == 3 ? 5 : 6; }
}  // namespace v3

// kbytes: bytes of K per row (kParts == 3, split fp32 rows: of one part).
struct TileSrc8 {
  u32x4 ra1, rg1, ra2, rg2;
  uint32_t roff_a[v3::kDma], roff_g[v3::kDma];
  int64_t kbytes_a, kbytes_g;
  bool live;                 // this wave's 64 x 64 block has live rows and columns
  int first = 0, count = 0;  // kPiece: the gradient stages this workgroup runs
};

__device__ __forceinline__ int dma_row8(int w, int j, int lane) { return 8 * (v3::kDma * w + j) + (lane >> 3); }

struct DmaState8 {
  u32x4 ra1, rg1, ra2, rg2;
  uint32_t roa[v3::kDma], rog[v3::kDma];
  uint32_t cbyte, lds0;
  int uwave, na, nst, first;
  int64_t kba, kbg;
};

// Instructions [j0, j1) of stage st's loads for this wave (6 per wave and
// stage).  Instruction j of wave w loads tile rows 8*(6w + j) .. +7 (rows <
// 256 are side 1); lane l -> row 8*(6w+j) + l/8, slot l%8 holding logical
// chunk (l%8) ^ (l/8), which is cbyte / 16.  A select between the four
// descriptors would be turned into a pointer select over stack copies (a
// scratch load, and the compiler then waits for every outstanding load before
// using it), so the descriptor is picked by mask arithmetic.
template <int kParts>
__device__ __forceinline__ void dma_part8(const DmaState8& D, int st, int j0, int j1) {
  const bool act = st < D.na;
  const int64_t kb = act ? D.kba : D.kbg;
  const int ks = act ? st : st - D.na + D.first;
  uint32_t koff1 = (uint32_t)ks * v2::kSB, koff2 = koff1;
  bool kin = st < D.nst;
  if constexpr (kParts == 3) {  // whole stages: no chunk past the width
    const split::Offsets o = split::offsets(ks, (int)(kb / v2::kSB), (uint32_t)kb);
    koff1 = o.k1;
    koff2 = o.k2;
  } else {
    kin = kin && (int64_t)(koff1 + D.cbyte) < kb;
  }
  const uint32_t base = D.lds0 + (uint32_t)((st % v2::kNBuf) * v2::kStage + v3::kDma * D.uwave * 8 * v2::kSB);
#pragma unroll
  for (int j = j0; j < j1; ++j) {
    const bool side1 = v3::kDma * D.uwave + j < v2::kBM / 8;  // uniform
    const uint32_t m = act ? 0xffffffffu : 0u;
    const uint32_t roff = (D.roa[j] & m) | (D.rog[j] & ~m);
    const uint32_t ms = side1 ? 0xffffffffu : 0u;
    u32x4 rs;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      rs[c] = (((D.ra1[c] & m) | (D.rg1[c] & ~m)) & ms) | (((D.ra2[c] & m) | (D.rg2[c] & ~m)) & ~ms);
    const uint32_t koff = side1 ? koff1 : koff2;
    dma16(rs, base + (uint32_t)(j * 8 * v2::kSB), (kin && roff != v2::kOob) ? roff + koff + D.cbyte : v2::kOob);
  }
}

// One slice: the 4 MFMAs of (ua, ub) into acc, with rd the 4 fragment reads
// of the slice two ahead (stage base sb, chunk offset coff) into (na, nb), and
// with qd >= 0 quarter qd's share of stage dst's loads (after MFMAs 1 and 3).
template <int DT, int kParts>
__device__ __forceinline__ void ghost_quarter8(f32x16 (&acc)[2][2], const u32x4 (&ua)[2], const u32x4 (&ub)[2],
                                               bool rd, const lds_char* sb, int coff, int wm, int wn,
                                               u32x4 (&na)[2], u32x4 (&nb)[2], const DmaState8& D, int qd, int dst) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (rd) {
      if (i < 2) na[i] = *(const u32x4*)(sb + (64 * wm + 32 * i) * v2::kSB + coff);
      else nb[i - 2] = *(const u32x4*)(sb + (v2::kBM + 64 * wn + 32 * (i - 2)) * v2::kSB + coff);
    }
    Mfma32<DT>::mma(acc[i >> 1][i & 1], ua[i >> 1], ub[i & 1]);
    if (qd >= 0 && i == 1) dma_part8<kParts>(D, dst, v3::lo(qd), v3::lo(qd) + 1);
    if (qd >= 0 && i == 3 && v3::lo(qd + 1) - v3::lo(qd) > 1) dma_part8<kParts>(D, dst, v3::lo(qd) + 1, v3::lo(qd + 1));
    __builtin_amdgcn_sched_barrier(0);
  }
}

__device__ __forceinline__ void ghost_stage_sync8() {
  static_assert(v2::kNBuf == 3, "vmcnt below is one stage of 6 instructions");
  asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);
  asm volatile("s_barrier" ::: "memory");
}

// Runs the tile's K stages; returns with every wave done reading the ring
// (so the caller may reuse the LDS) and no load in flight.
// kHasA: the tile has activation stages (K > 0), multiplied into ka before
// the gradient stages into kg; otherwise every stage goes to kg and ka stays 0.
// kPiece (without kHasA): only the stages [S.first, S.first + S.count).
// Fragment offsets inside a stage: A fragment x = rows 64wm + 32x + l%32, B
// fragment y = rows 256 + 64wn + 32y + l%32; slice kk reads logical chunk
// 2kk + l/32, stored in slot (2kk + l/32) ^ (l%8).  Fragments are read two
// slices ahead of their MFMAs, so a read has a whole slice of MFMAs to come
// back while the DMA writes share the LDS.  A loop body starts right after a
// barrier (no read in flight, so the loop header needs no wait): it
// multiplies slices 2 and 3 of stage st and slices 0 and 1 of st + 1 while
// reading slices 0..3 of st + 1, loads stage st + 3 into the buffer stage st
// left (its reads all ended before that barrier), then waits for stage st + 2.
// Exactly the 6 instructions of the body's own loads follow the awaited
// stage's last one at every barrier.  A wave without live rows or columns
// passes the same barriers with the same loads.
template <int DT, bool kHasA, int kParts, bool kPiece = false>
__device__ __forceinline__ void ghost_tile_engine8(const TileSrc8& S, char* smem, f32x16 (&ka)[2][2],
                                                   f32x16 (&kg)[2][2]) {
  lds_char* const L = (lds_char*)smem;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  DmaState8 D;
  D.uwave = __builtin_amdgcn_readfirstlane(wave);
  constexpr int kSegs = kParts == 3 ? split::kSegs : 1;
  D.na = kSegs * (int)((S.kbytes_a + v2::kSB - 1) / v2::kSB);
  D.nst = kPiece ? S.count : D.na + kSegs * (int)((S.kbytes_g + v2::kSB - 1) / v2::kSB);
  D.first = kPiece ? S.first : 0;
  D.ra1 = uniform4(S.ra1);
  D.rg1 = uniform4(S.rg1);
  D.ra2 = uniform4(S.ra2);
  D.rg2 = uniform4(S.rg2);
  D.kba = S.kbytes_a;
  D.kbg = S.kbytes_g;
  D.lds0 = (uint32_t)(uintptr_t)L;
  D.cbyte = 16u * (uint32_t)((lane & 7) ^ (lane >> 3));
#pragma unroll
  for (int j = 0; j < v3::kDma; ++j) {
    D.roa[j] = S.roff_a[j];
    D.rog[j] = S.roff_g[j];
  }
  const int na = D.na, nst = D.nst;
  if (!__builtin_amdgcn_readfirstlane((int)S.live)) {  // products of zero rows: this wave's loads and barriers only
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) ka[x][y] = kg[x][y] = f32x16{};
    dma_part8<kParts>(D, 0, 0, v3::kDma);
    for (int st = 0; st <= max(nst, 1); ++st) {
      dma_part8<kParts>(D, st + 1, 0, v3::kDma);
      ghost_stage_sync8();
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    return;
  }

  const int lrow = lane & 31, hh = lane >> 5;
  const int c0 = lrow * v2::kSB + (((0 + hh) ^ (lane & 7)) << 4), c1 = lrow * v2::kSB + (((2 + hh) ^ (lane & 7)) << 4);
  const int c2 = lrow * v2::kSB + (((4 + hh) ^ (lane & 7)) << 4), c3 = lrow * v2::kSB + (((6 + hh) ^ (lane & 7)) << 4);
  u32x4 fa[4][2], fb[4][2];

#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      ka[x][y] = f32x16{};
      kg[x][y] = f32x16{};
    }

#pragma unroll
  for (int s0 = 0; s0 < v2::kNBuf - 1; ++s0) dma_part8<kParts>(D, s0, 0, v3::kDma);
  ghost_stage_sync8();
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const int co = kk == 0 ? c0 : c1;
#pragma unroll
    for (int x = 0; x < 2; ++x) fa[kk][x] = *(const u32x4*)(L + (64 * wm + 32 * x) * v2::kSB + co);
#pragma unroll
    for (int y = 0; y < 2; ++y) fb[kk][y] = *(const u32x4*)(L + (v2::kBM + 64 * wn + 32 * y) * v2::kSB + co);
  }
  dma_part8<kParts>(D, v2::kNBuf - 1, v3::lo(0), v3::lo(2));
  {
    f32x16(&acc0)[2][2] = kHasA ? ka : kg;
    ghost_quarter8<DT, kParts>(acc0, fa[0], fb[0], true, L, c2, wm, wn, fa[2], fb[2], D, 2, v2::kNBuf - 1);
    ghost_quarter8<DT, kParts>(acc0, fa[1], fb[1], true, L, c3, wm, wn, fa[3], fb[3], D, 3, v2::kNBuf - 1);
  }
  ghost_stage_sync8();

#define DA_GHOST_BODY8(A1, A2)                                                                        \
  {                                                                                                   \
    const lds_char* nxt = L + ((st + 1) % v2::kNBuf) * v2::kStage;                                    \
    ghost_quarter8<DT, kParts>(A1, fa[2], fb[2], true, nxt, c0, wm, wn, fa[0], fb[0], D, 0, st + 3);          \
    ghost_quarter8<DT, kParts>(A1, fa[3], fb[3], true, nxt, c1, wm, wn, fa[1], fb[1], D, 1, st + 3);          \
    ghost_quarter8<DT, kParts>(A2, fa[0], fb[0], true, nxt, c2, wm, wn, fa[2], fb[2], D, 2, st + 3);          \
    ghost_quarter8<DT, kParts>(A2, fa[1], fb[1], true, nxt, c3, wm, wn, fa[3], fb[3], D, 3, st + 3);          \
    ghost_stage_sync8();                                                                              \
  }
  if constexpr (kHasA) {
    for (int st = 0; st + 1 < na; ++st) DA_GHOST_BODY8(ka, ka)
    {
      const int st = na - 1;
      DA_GHOST_BODY8(ka, kg)
    }
  }
  for (int st = kHasA ? na : 0; st + 1 < nst; ++st) DA_GHOST_BODY8(kg, kg)
#undef DA_GHOST_BODY8
  ghost_quarter8<DT, kParts>(kg, fa[2], fb[2], false, L, c0, wm, wn, fa[0], fb[0], D, -1, 0);
  ghost_quarter8<DT, kParts>(kg, fa[3], fb[3], false, L, c1, wm, wn, fa[1], fb[1], D, -1, 0);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Dense / per-sample segmented mode: a 256 x 128 tile inside one sample pair on
// the 8-wave engine.  Its fp32 partial (the 8 waves' shares summed in a fixed
// order) goes to the pair's slot; ghost_gram_reduce adds a pair's tiles.
template <int DT, int kParts = 1>
__global__ __launch_bounds__(v3::kThreads, 1) void ghost_gram_tiles_v3(GhostArgs g) {
  __shared__ __attribute__((aligned(1024))) char smem[v2::kRing];
  __shared__ float red[v3::kWaves];
  if (gate_closed(g.gate)) return;
  // Each XCD runs 32 tiles at once; grouping 4 row tiles (4 MB of operand rows
  // each at d = 4096) with 8 column tiles (2 MB each) minimises the rows its L2
  // streams per block of concurrent tiles (measured: groups of 4 rows beat 8,
  // 16 and 32 by 6%, 17% and 40% on the 256 x 64 pair, T = 512 workload).
  constexpr int64_t kRowGroup = 4;
  const int64_t logical = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t per_group = kRowGroup * g.n_c;
  const int64_t group = logical / per_group;
  const int64_t first_r = group * kRowGroup;
  const int64_t gsize = min(g.n_r - first_r, kRowGroup);
  const int64_t in_group = logical - group * per_group;
  const int64_t R = first_r + in_group % gsize;
  const int64_t C = in_group / gsize;
  const int64_t i = R / g.tiles_r, tt = R % g.tiles_r;
  const int64_t j = pair_col_sample(g, i, C), ss = C % g.tiles_c;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  const int64_t len1 = seg_len(g.s1, i), len2 = seg_len(g.s2, j);
  const int64_t t0 = tt * v2::kBM, s0 = ss * v2::kBN;
  float* dst = g.partial + (pair_slot(g, i, j) * g.tiles_r + tt) * g.tiles_c + ss;
  if (t0 >= len1 || s0 >= len2) {
    if (tid == 0) *dst = 0.f;
    return;
  }
  const int64_t st1 = seg_start(g.s1, i), st2 = seg_start(g.s2, j);
  // Buffer bases: the sample's first row (dense) or the factor (segmented);
  // the host checked that every offset stays below 2^31.
  const char* ba1 = g.s1.seg ? g.s1.act : g.s1.act + i * g.s1.act_bstride;
  const char* bg1 = g.s1.seg ? g.s1.grad : g.s1.grad + i * g.s1.grad_bstride;
  const char* ba2 = g.s2.seg ? g.s2.act : g.s2.act + j * g.s2.act_bstride;
  const char* bg2 = g.s2.seg ? g.s2.grad : g.s2.grad + j * g.s2.grad_bstride;
  TileSrc8 S;
  S.ra1 = make_rsrc(ba1, 0x7fffffffu);
  S.rg1 = make_rsrc(bg1, 0x7fffffffu);
  S.ra2 = make_rsrc(ba2, 0x7fffffffu);
  S.rg2 = make_rsrc(bg2, 0x7fffffffu);
  S.kbytes_a = g.kbytes_a;
  S.kbytes_g = g.kbytes_g;
  S.live = t0 + 64 * (wave >> 1) < len1 && s0 + 64 * (wave & 1) < len2;
#pragma unroll
  for (int q = 0; q < v3::kDma; ++q) {
    const int row = dma_row8(wave, q, lane);
    const bool side1 = row < v2::kBM;
    const SideDev& sd = side1 ? g.s1 : g.s2;
    const int64_t t = side1 ? t0 + row : s0 + row - v2::kBM;
    const int64_t len = side1 ? len1 : len2;
    const int64_t start = side1 ? st1 : st2;
    if (t < len) {
      const int64_t r = sd.seg ? (sd.idx ? (int64_t)sd.idx[start + t] : start + t) : t;
      S.roff_a[q] = (uint32_t)(r * sd.act_tstride);
      S.roff_g[q] = (uint32_t)(r * sd.grad_tstride);
    } else {
      S.roff_a[q] = v2::kOob;
      S.roff_g[q] = v2::kOob;
    }
  }
  f32x16 ka[2][2], kg[2][2];
  ghost_tile_engine8<DT, true, kParts>(S, smem, ka, kg);
  float s = 0.f;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) s += (ka[x][y][r] + g.bias) * kg[x][y][r];
  s = wave_sum(s);
  if (lane == 0) red[wave] = s;
  __syncthreads();
  if (tid == 0) *dst = ((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7]));
}

// Grouped (MoE) mode: tiles over each group's packed rows, the tile's
// products parked in LDS and binned by sample pair.  One workgroup fits a CU,
// so tiles run in rounds of as many as there are CUs, and what is left after
// the last full round would hold the chip for a whole tile's time: those tiles
// run in pieces (stage ranges of one of the two products, all tiles' pieces of
// one range together so that they share operand rows in L2), each leaving its
// fp32 accumulators in the workspace for ghost_grouped_finish.
template <int DT, int kParts = 1>
__global__ __launch_bounds__(v3::kThreads, 1) void ghost_grouped_tiles_v3(GroupedArgs ga) {
  __shared__ __attribute__((aligned(1024))) char smem[v2::kSmem];
  if (gate_closed(ga.gate)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  // Tiles go to the XCDs round-robin in launch order (no XCD remap): the host
  // orders the groups longest reduction first, so every XCD gets the same mix
  // of tile lengths, longest first.  A contiguous range per XCD would hand the
  // long groups' tiles to some XCDs and the short ones to the rest; consecutive
  // tiles of every round of 256 per XCD measured the same (1102 tiles of 360
  // stages 1715 against 1728 us, 8 experts' tiles 1081 either way).
  const bool piece = (int)blockIdx.x >= ga.whole;
  int32_t local = (int32_t)blockIdx.x - (piece ? ga.whole : 0);
  int e = 0;
  while (e + 1 < ga.n_groups && (piece ? ga.grp[e + 1].piece0 : ga.grp[e + 1].tile0) <= local) ++e;
  const GroupDev& G = ga.grp[e];
  int range = 0;
  const int32_t at_piece = local;
  if (piece) {
    const int32_t split = G.tiles_r * G.tiles_c - G.whole;
    local -= G.piece0;
    range = local / split;
    local = G.whole + local - range * split;
  } else {
    local -= G.tile0;
  }
  int32_t m, n;
  group_tile<kTileRows>(G, local, m, n);

  const int64_t t0 = (int64_t)m * v2::kBM, s0 = (int64_t)n * v2::kBN;
  // Rows at or past seg[B] belong to no sample (and may have no row_index
  // entry); a tile wholly past the packed rows of a side owns no bin.
  const int64_t n1 = min(G.rows1, (int64_t)G.seg1[ga.b1]), n2 = min(G.rows2, (int64_t)G.seg2[ga.b2]);
  if (t0 >= n1 || s0 >= n2) return;
  TileSrc8 S;
  S.ra1 = make_rsrc(G.a1, 0x7fffffffu);
  S.rg1 = make_rsrc(G.g1, 0x7fffffffu);
  S.ra2 = make_rsrc(G.a2, 0x7fffffffu);
  S.rg2 = make_rsrc(G.g2, 0x7fffffffu);
  S.kbytes_a = G.kbytes_a;
  S.kbytes_g = G.kbytes_g;
  S.live = t0 + 64 * wm < n1 && s0 + 64 * wn < n2;
#pragma unroll
  for (int q = 0; q < v3::kDma; ++q) {
    const int row = dma_row8(wave, q, lane);
    const bool side1 = row < v2::kBM;
    const int64_t t = side1 ? t0 + row : s0 + row - v2::kBM;
    const bool live = t < (side1 ? n1 : n2);
    const int32_t* idx = side1 ? G.idx1 : G.idx2;
    const int64_t r = live ? (idx ? (int64_t)idx[t] : t) : 0;
    S.roff_a[q] = live ? (uint32_t)(r * (side1 ? G.a1_ts : G.a2_ts)) : v2::kOob;
    S.roff_g[q] = live ? (uint32_t)(r * (side1 ? G.g1_ts : G.g2_ts)) : v2::kOob;
  }
  f32x16 ka[2][2], kg[2][2];
  if (piece) {
    const bool act = range < G.pieces_a;
    const int np = act ? G.pieces_a : G.pieces_g, at = act ? range : range - G.pieces_a;
    if (act) {
      S.rg1 = S.ra1;
      S.rg2 = S.ra2;
      S.kbytes_g = S.kbytes_a;
#pragma unroll
      for (int q = 0; q < v3::kDma; ++q) S.roff_g[q] = S.roff_a[q];
    }
    const int stages = (kParts == 3 ? split::kSegs : 1) * (int)((S.kbytes_g + v2::kSB - 1) / v2::kSB);
    S.kbytes_a = 0;
    S.first = stages * at / np;
    S.count = stages * (at + 1) / np - S.first;
    ghost_tile_engine8<DT, false, kParts, true>(S, smem, ka, kg);
    f32x4* d = (f32x4*)(ga.dump + (int64_t)at_piece * kPieceFloats) + tid;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          d[((x * 2 + y) * 4 + q) * v3::kThreads] =
              f32x4{kg[x][y][4 * q], kg[x][y][4 * q + 1], kg[x][y][4 * q + 2], kg[x][y][4 * q + 3]};
    return;
  }
  ghost_tile_engine8<DT, true, kParts>(S, smem, ka, kg);
  float* P = (float*)smem;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 64 * wm + 32 * x + acc_row(r, lane), col = 64 * wn + 32 * y + acc_col(lane);
        P[row * v2::kPRow + col] = (ka[x][y][r] + G.bias) * kg[x][y][r];
      }
  __syncthreads();
  pair_bins<64>(P, v2::kPRow, t0, s0, n1, n2, m, n, G, ga, ga.partial + G.part_off);
}

// The split tiles: one workgroup adds the pieces of a 64-row slab (in order,
// the activation product's, then the gradient one's), multiplies and bins.
// Thread (lane, q): the four accumulators 4q .. 4q + 3 of each 32 x 32 block as
// lane `lane` of the two waves that own the slab held them.
constexpr int kFinishThreads = 256;
__global__ __launch_bounds__(kFinishThreads) void ghost_grouped_finish(GroupedArgs ga) {
  __shared__ float P[kSlab * kPRow];
  if (gate_closed(ga.gate)) return;
  constexpr int kSlabs = v2::kBM / kSlab;
  int32_t local = (int32_t)(blockIdx.x / kSlabs);
  const int wm = (int)(blockIdx.x % kSlabs);
  int e = 0;
  for (; e + 1 < ga.n_groups; ++e) {
    const int32_t split = ga.grp[e].tiles_r * ga.grp[e].tiles_c - ga.grp[e].whole;
    if (local < split) break;
    local -= split;
  }
  const GroupDev& G = ga.grp[e];
  const int32_t split = G.tiles_r * G.tiles_c - G.whole;
  int32_t m, n;
  group_tile<kTileRows>(G, G.whole + local, m, n);
  const int64_t n1 = min(G.rows1, (int64_t)G.seg1[ga.b1]), n2 = min(G.rows2, (int64_t)G.seg2[ga.b2]);
  const int64_t t0 = (int64_t)m * v2::kBM + wm * kSlab, s0 = (int64_t)n * v2::kBN;
  if (t0 >= n1 || s0 >= n2) return;
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int64_t stride = (int64_t)split * kPieceFloats / 4;
#pragma unroll
  for (int wn = 0; wn < 2; ++wn) {
    const f32x4* src = (const f32x4*)ga.dump + (int64_t)(G.piece0 + local) * (kPieceFloats / 4) +
                       q * v3::kThreads + (2 * wm + wn) * kWave + lane;
    f32x4 k[2][4];  // the two products of blocks (x, y) = (b / 2, b % 2)
#pragma unroll
    for (int b = 0; b < 4; ++b) k[0][b] = k[1][b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int np = h ? G.pieces_g : G.pieces_a;
#pragma unroll 4
      for (int p = 0; p < np; ++p, src += stride)
#pragma unroll
        for (int b = 0; b < 4; ++b) k[h][b] += src[b * 4 * v3::kThreads];
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 32 * (b >> 1) + acc_row(4 * q + r, lane), col = 64 * wn + 32 * (b & 1) + acc_col(lane);
        P[row * kPRow + col] = (k[0][b][r] + G.bias) * k[1][b][r];
      }
  }
  __syncthreads();
  pair_bins<kSlab / 2>(P, kPRow, t0, s0, n1, n2, (int64_t)m * kSlabs + wm, n, G, ga, ga.partial + G.slab_off);
}

// ---------------------------------------------------------------------------
// Per-token cross-gram on the 256 x 128 engine: K[i, t, j] keeps side 1's
// token t and sums side 2 out (the token decomposition of the score).
//
//   factorized side 2:  K[i,t,j] = sum_s (a1_it . a2_js + bias)(g1_it . g2_js)
//   dense side 2:       K[i,t,j] = sum_o (a1_it . M2_j[o,:] + mb_j[o]) g1_it[o]
//
// The factorized form is the ghost tile with a row epilogue; the dense form
// runs the engine's second product alone over a1 rows against M2_j's rows (the
// output channels o play side 2's tokens) and multiplies by g1 in the
// epilogue.  Each tile parks its (256 x 128) products in LDS and sums every
// row over its 128 columns; a second kernel adds the column tiles in order.
// ---------------------------------------------------------------------------
struct PerTokArgs {
  SideDev s1, s2;                  // dense form: s2.grad = M2 rows (tokens = D)
  int64_t kbytes_a, kbytes_g;
  int64_t tiles_r, tiles_c, n_r, n_c;
  float bias;                      // factorized: the implicit ones column
  const float* m2bias;             // dense: (B2, D) fp32 bias-column gradients, or nullptr
  int64_t m2bias_ld;               // floats between samples
  int64_t tpad;                    // tiles_r * 256
  float* partial;                  // [B1][B2][tpad][tiles_c]
  Gate gate;
};

template <int DT, bool kDense, int kParts = 1>
__global__ __launch_bounds__(v3::kThreads, 1) void ghost_per_token_v3(PerTokArgs g) {
  static_assert(!kDense || kParts == 1, "the dense epilogue reads g1 in DT");
  __shared__ __attribute__((aligned(1024))) char smem[v2::kSmem];
  if (gate_closed(g.gate)) return;
  constexpr int64_t kRowGroup = 4;
  const int64_t logical = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t per_group = kRowGroup * g.n_c;
  const int64_t group = logical / per_group;
  const int64_t first_r = group * kRowGroup;
  const int64_t gsize = min(g.n_r - first_r, kRowGroup);
  const int64_t in_group = logical - group * per_group;
  const int64_t R = first_r + in_group % gsize;
  const int64_t C = in_group / gsize;
  const int64_t i = R / g.tiles_r, tt = R % g.tiles_r;
  const int64_t j = C / g.tiles_c, ss = C % g.tiles_c;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t len1 = g.s1.tokens, len2 = g.s2.tokens;
  const int64_t t0 = tt * v2::kBM, s0 = ss * v2::kBN;
  if (t0 >= len1) return;  // uniform: no row of this tile is read back
  TileSrc8 S;
  S.ra1 = make_rsrc(g.s1.act + i * g.s1.act_bstride, 0x7fffffffu);
  S.rg1 = make_rsrc((kDense ? g.s1.act : g.s1.grad) + i * (kDense ? g.s1.act_bstride : g.s1.grad_bstride),
                    0x7fffffffu);
  S.ra2 = make_rsrc(g.s2.grad + j * g.s2.grad_bstride, 0x7fffffffu);
  S.rg2 = make_rsrc(g.s2.grad + j * g.s2.grad_bstride, 0x7fffffffu);
  if (!kDense) S.ra2 = make_rsrc(g.s2.act + j * g.s2.act_bstride, 0x7fffffffu);
  S.kbytes_a = g.kbytes_a;
  S.kbytes_g = g.kbytes_g;
  // 16-bit rows: edge tiles are bound by their loads, and the choice costs full ones 0.5%.
  S.live = (DT != DA_F32 && kParts == 1) || (t0 + 64 * wm < len1 && s0 + 64 * wn < len2);
#pragma unroll
  for (int q = 0; q < v3::kDma; ++q) {
    const int row = dma_row8(wave, q, lane);
    const bool side1 = row < v2::kBM;
    const int64_t t = side1 ? t0 + row : s0 + row - v2::kBM;
    if (t < (side1 ? len1 : len2)) {
      // dense form: side 1 streams a1 rows and side 2 M2_j rows, both in the gradient loop
      const int64_t ts1 = kDense ? g.s1.act_tstride : g.s1.grad_tstride;
      S.roff_a[q] = (uint32_t)(t * (side1 ? g.s1.act_tstride : g.s2.act_tstride));
      S.roff_g[q] = (uint32_t)(t * (side1 ? ts1 : g.s2.grad_tstride));
    } else {
      S.roff_a[q] = v2::kOob;
      S.roff_g[q] = v2::kOob;
    }
  }
  f32x16 ka[2][2], kg[2][2];
  ghost_tile_engine8<DT, !kDense, kParts>(S, smem, ka, kg);
  float* P = (float*)smem;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 64 * wm + 32 * x + acc_row(r, lane), col = 64 * wn + 32 * y + acc_col(lane);
        float v;
        if constexpr (kDense) {
          const int64_t t = t0 + row, o = s0 + col;
          const bool ok = t < len1 && o < len2;
          const float gv = ok ? Elem<DT>::load(g.s1.grad + i * g.s1.grad_bstride + t * g.s1.grad_tstride, o) : 0.f;
          const float mb = (ok && g.m2bias) ? g.m2bias[j * g.m2bias_ld + o] : 0.f;
          v = (kg[x][y][r] + mb) * gv;
        } else {
          v = (ka[x][y][r] + g.bias) * kg[x][y][r];
        }
        P[row * v2::kPRow + col] = v;
      }
  __syncthreads();
  // one thread per row: the row's 128 columns in order (zero past side 2's end)
  const int64_t t = t0 + tid;
  if (tid < v2::kBM && t < len1) {
    const float* pr = P + tid * v2::kPRow;
    float sum = 0.f;
    for (int c = 0; c < v2::kBN; ++c) sum += pr[c];
    g.partial[((i * g.s2.batch + j) * g.tpad + t) * g.tiles_c + ss] = sum;
  }
}

// out[i*ld_b1 + t*ld_t + j*ld_b2] (+)= sum over column tiles, in order.
__global__ void per_token_reduce(const float* __restrict__ partial, int64_t b1, int64_t len1, int64_t b2,
                                 int64_t tpad, int64_t tiles_c, float* __restrict__ out, int64_t ld_b1,
                                 int64_t ld_t, int64_t ld_b2, int accumulate) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= b1 * len1 * b2) return;
  const int64_t j = idx % b2, t = (idx / b2) % len1, i = idx / (b2 * len1);
  const float* p = partial + ((i * b2 + j) * tpad + t) * tiles_c;
  float s = 0.f;
  for (int64_t q = 0; q < tiles_c; ++q) s += p[q];
  float* o = out + i * ld_b1 + t * ld_t + j * ld_b2;
  *o = accumulate ? *o + s : s;
}

struct Plan {
  int64_t tiles_r, tiles_c, n_r, n_c, per_pair;
  size_t ws;
  bool v2;  // the 256 x 128 tile engine (dense sides whose offsets fit 31 bits, D > 0)
  size_t split_ws;  // bytes behind ws for the split copies of fp32 factors; 0: not split
};

// The tile engine addresses a sample's rows with 32-bit buffer offsets.
bool fits_v2(const da_factor_side* s, int64_t K, int64_t D, int64_t es) {
  if (s->seg_offsets) return false;
  const int64_t ts = s->act_tstride > s->grad_tstride ? s->act_tstride : s->grad_tstride;
  const int64_t w = K > D ? K : D;
  return s->act_tstride >= 0 && s->grad_tstride >= 0 && (s->tokens * ts + w) * es < (1LL << 31) - (1LL << 20);
}

size_t align256(size_t n) { return (n + 255) / 256 * 256; }

// Bytes of a call's split copies (0: the call stays on fp32 rows): dense sides
// on the tile engine, `tiles` of them, whose split rows its 32-bit offsets reach.
size_t split_sides(const da_factor_side* s1, const da_factor_side* s2, int64_t K, int64_t D, int64_t tiles) {
  const da_factor_side* sides[2] = {s1, s2};
  const int64_t ts = split::row_bytes(K > D ? K : D), lim = (1LL << 31) - (1LL << 20);
  int64_t slots = 0;
  if (device_cu_count(&slots) != DA_OK) return 0;
  split::Cost cost;
  size_t bytes = 256;
  for (const da_factor_side* s : sides) {
    const int64_t rows = s->batch * s->tokens;
    if ((s->tokens + 1) * ts >= lim) return 0;
    bytes += split::Builder::bytes(rows, K) + split::Builder::bytes(rows, D);
    cost.values += (double)rows * (double)(K + D);
  }
  cost.tiles((double)tiles, K, 4.0);
  cost.tiles((double)tiles, D, 4.0);
  cost.end_chain();
  return bytes <= split::kMaxBytes && cost.pays(slots) ? bytes : 0;
}

// A dense side's factors split into `b`: the side as the 2-byte engine reads it.
SideDev split_side(split::Builder& b, const SideDev& s, int64_t K, int64_t D) {
  SideDev d = s;
  d.act = b.add(s.act, s.batch, s.tokens, s.act_bstride, s.act_tstride, K);
  d.grad = b.add(s.grad, s.batch, s.tokens, s.grad_bstride, s.grad_tstride, D);
  d.act_tstride = split::row_bytes(K);
  d.grad_tstride = split::row_bytes(D);
  d.act_bstride = s.tokens * d.act_tstride;
  d.grad_bstride = s.tokens * d.grad_tstride;
  return d;
}

int validate_side(const da_factor_side* s, int64_t K, int64_t D, int dtype, const char* name) {
  if (!s) return set_error(DA_ERR_INVALID, "da_ghost_gram: %s is NULL", name);
  if (s->batch < 0 || s->tokens < 0)
    return set_error(DA_ERR_INVALID, "da_ghost_gram: %s has negative batch/tokens", name);
  if (s->batch == 0 || s->tokens == 0) return DA_OK;
  if (!s->act || !s->grad) return set_error(DA_ERR_INVALID, "da_ghost_gram: %s has NULL factor", name);
  const int64_t es = (int64_t)elem_bytes(dtype);
  if (((uintptr_t)s->act | (uintptr_t)s->grad) & 15)
    return set_error(DA_ERR_INVALID, "da_ghost_gram: %s factors must be 16-byte aligned", name);
  const int64_t strides[4] = {s->act_bstride, s->act_tstride, s->grad_bstride, s->grad_tstride};
  for (int q = 0; q < 4; ++q) {
    if (s->seg_offsets && (q == 0 || q == 2)) continue;  // batch strides unused when segmented
    if ((strides[q] * es) % 16)
      return set_error(DA_ERR_INVALID, "da_ghost_gram: %s strides must be multiples of 16 bytes", name);
  }
  (void)K;
  (void)D;
  return DA_OK;
}

int make_plan(const da_factor_side* s1, const da_factor_side* s2, int64_t K, int64_t D, int dtype,
              Plan* plan, bool diag = false) {
  if (!valid_dtype(dtype)) return set_error(DA_ERR_INVALID, "da_ghost_gram: bad dtype %d", dtype);
  if (K < 0 || D < 0) return set_error(DA_ERR_INVALID, "da_ghost_gram: negative width");
  const int64_t es = (int64_t)elem_bytes(dtype);
  if ((K * es) % 16 || (D * es) % 16)
    return set_error(DA_ERR_INVALID,
                     "da_ghost_gram: K=%lld and D=%lld must be multiples of %lld elements",
                     (long long)K, (long long)D, (long long)(16 / es));
  int rc = validate_side(s1, K, D, dtype, "s1");
  if (rc) return rc;
  rc = validate_side(s2, K, D, dtype, "s2");
  if (rc) return rc;
  if (s1->has_bias != s2->has_bias)
    return set_error(DA_ERR_INVALID, "da_ghost_gram: both sides must agree on has_bias");
  plan->v2 = fits_v2(s1, K, D, es) && fits_v2(s2, K, D, es) && D > 0 && K > 0;
  const int64_t bm = plan->v2 ? v2::kBM : kBM, bn = plan->v2 ? v2::kBN : kBN;
  plan->tiles_r = (s1->tokens + bm - 1) / bm;
  plan->tiles_c = (s2->tokens + bn - 1) / bn;
  if (diag && s1->batch != s2->batch)
    return set_error(DA_ERR_INVALID, "da_ghost_gram_diag: the two sides need one batch size (%lld vs %lld)",
                     (long long)s1->batch, (long long)s2->batch);
  plan->n_r = s1->batch * plan->tiles_r;
  plan->n_c = (diag ? 1 : s2->batch) * plan->tiles_c;
  plan->per_pair = plan->tiles_r * plan->tiles_c;
  plan->ws = (size_t)(s1->batch * (diag ? 1 : s2->batch) * plan->per_pair) * sizeof(float);
  plan->split_ws = 0;
  if (dtype == DA_F32 && plan->v2) {
    plan->split_ws = split_sides(s1, s2, K, D, plan->n_r * plan->n_c);
    if (plan->split_ws) plan->ws = align256(plan->ws);
  }
  return DA_OK;
}

SideDev to_dev(const da_factor_side* s, int64_t es) {
  SideDev d;
  d.act = (const char*)s->act;
  d.grad = (const char*)s->grad;
  d.batch = s->batch;
  d.tokens = s->tokens;
  d.act_bstride = s->act_bstride * es;
  d.act_tstride = s->act_tstride * es;
  d.grad_bstride = s->grad_bstride * es;
  d.grad_tstride = s->grad_tstride * es;
  d.seg = s->seg_offsets;
  d.idx = s->row_index;
  return d;
}


// Per-token plans.  Both forms need dense sides (one row range per sample)
// whose rows the 256 x 128 engine addresses with 32-bit offsets.
struct PerTokPlan {
  int64_t tiles_r, tiles_c, tpad;
  size_t ws;
  size_t split_ws;  // bytes behind ws for the split copies of fp32 factors; 0: not split
};

// The factorized form's split copies, once both sides are known to be dense.
void per_token_split(const da_factor_side* s1, const da_factor_side* s2, int64_t K, int64_t D, int dtype,
                     PerTokPlan* p) {
  if (dtype != DA_F32 || K <= 0 || D <= 0 || s1->batch <= 0 || s1->tokens <= 0 || s2->batch <= 0 || s2->tokens <= 0 || !fits_v2(s1, K, D, 4) || !fits_v2(s2, K, D, 4)) return;
  p->split_ws = split_sides(s1, s2, K, D, s1->batch * p->tiles_r * s2->batch * p->tiles_c);
  if (p->split_ws) p->ws = align256(p->ws);
}

int per_token_plan(const da_factor_side* s1, int64_t b2, int64_t len2, int64_t K, int64_t D, int dtype,
                   const char* who, PerTokPlan* p) {
  if (!valid_dtype(dtype)) return set_error(DA_ERR_INVALID, "%s: bad dtype %d", who, dtype);
  if (K < 0 || D < 0 || b2 < 0 || len2 < 0) return set_error(DA_ERR_INVALID, "%s: negative size", who);
  const int64_t es = (int64_t)elem_bytes(dtype);
  if ((K * es) % 16 || (D * es) % 16)
    return set_error(DA_ERR_INVALID, "%s: K=%lld and D=%lld must be multiples of %lld elements", who,
                     (long long)K, (long long)D, (long long)(16 / es));
  if (!s1) return set_error(DA_ERR_INVALID, "%s: s1 is NULL", who);
  p->tiles_r = (s1->tokens + v2::kBM - 1) / v2::kBM;
  p->tiles_c = (len2 + v2::kBN - 1) / v2::kBN;
  p->tpad = p->tiles_r * v2::kBM;
  p->ws = (size_t)(s1->batch * b2 * p->tpad * p->tiles_c) * sizeof(float);
  p->split_ws = 0;
  return DA_OK;
}

int per_token_launch(const PerTokArgs& g, bool dense, int dtype, int64_t len1, float* out, int64_t ld_b1,
                     int64_t ld_t, int64_t ld_b2, int accumulate, hipStream_t st, const char* who) {
  const int64_t tiles = g.n_r * g.n_c;
  if (tiles > 0x7fffffffLL) return set_error(DA_ERR_INVALID, "%s: problem too large", who);
#define DA_PT(DT)                                                                  \
  if (dense)                                                                       \
    ghost_per_token_v3<DT, true><<<(unsigned)tiles, v3::kThreads, 0, st>>>(g);     \
  else                                                                             \
    ghost_per_token_v3<DT, false><<<(unsigned)tiles, v3::kThreads, 0, st>>>(g);
  switch (dtype) {
    case DA_BF16: DA_PT(DA_BF16) break;
    case DA_F16: DA_PT(DA_F16) break;
    default: DA_PT(DA_F32) break;
  }
#undef DA_PT
  int rc = check_launch(who);
  if (rc) return rc;
  const int64_t n = g.s1.batch * len1 * g.s2.batch;
  per_token_reduce<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(g.partial, g.s1.batch, len1, g.s2.batch, g.tpad,
                                                                g.tiles_c, out, ld_b1, ld_t, ld_b2, accumulate);
  return check_launch(who);
}
}  // namespace
}  // namespace da

namespace da {
namespace {

struct GroupedPlan {
  size_t part_floats, ws;
  size_t split_ws; // bytes behind ws for the split copies of fp32 factors; 0: not split
  size_t tail_ws;  // bytes behind both for the tiles that run in pieces; 0: none
  bool v2;         // all groups on the 256 x 128 engine
  int tile_r, tile_c;
};

// A group of a launch as the tail planner sees it, longest reduction first.
struct TailGroup {
  int64_t tiles, na, ng;     // tiles, stages of the two products
  int64_t whole;             // out: tiles that run whole
  int pieces_a, pieces_g;    // out: pieces of each of the others
};

// Which of a launch's tiles run in pieces.  Full rounds run whole (groups of
// about one length share rounds: a shorter group's tiles do not fill a longer
// one's last round well); the rest, less than a round, is cut into pieces of at
// most p stages, one or two rounds of them, when that is expected to be faster.
// A stage takes stage_us; a piece about 2 us to start and to write its
// accumulators, which move twice at about 4 TB/s, and the finishing launch 6 us.
// Measured, whole tiles against this: 48 x 24 samples of 201 x 150 tokens, 768 ->
// 3072 in fp32 (1102 tiles of 360 stages) 1867 and 1647 us; 8 experts of about
// 1024 rows a side, 4096 -> 28672 and 14336 -> 4096 in bf16 (about 610 tiles)
// 1150 and 1063 us with their routing.
// Returns the number of pieces.
int64_t plan_tails(TailGroup* g, int n, int64_t slots, double stage_us) {
  auto chain = [&](int e) { return g[e].na + g[e].ng; };
  auto take = [&](int from, int to, int64_t count) {
    for (int e = from; e < to && count > 0; ++e) {
      const int64_t w = std::min(count, g[e].tiles - g[e].whole);
      g[e].whole += w;
      count -= w;
    }
  };
  for (int e = 0; e < n; ++e) g[e].whole = g[e].pieces_a = g[e].pieces_g = 0;
  for (int from = 0; from < n;) {
    int to = from;
    int64_t tiles = 0;
    while (to < n && 5 * chain(to) >= 4 * chain(from)) tiles += g[to++].tiles;
    take(from, to, tiles / slots * slots);
    from = to;
  }
  int64_t rest = 0, longest = 0, most = 0;
  for (int e = 0; e < n; ++e) rest += g[e].tiles - g[e].whole;
  take(0, n, rest / slots * slots);
  rest %= slots;
  for (int e = 0; e < n; ++e)
    if (g[e].tiles > g[e].whole) {
      longest = std::max(longest, chain(e));
      most = std::max(most, std::max(g[e].na, g[e].ng));
    }
  auto pieces = [&](int64_t p) {
    int64_t c = 0;
    for (int e = 0; e < n; ++e)
      c += (g[e].tiles - g[e].whole) * ((g[e].na + p - 1) / p + (g[e].ng + p - 1) / p);
    return c;
  };
  double best = 0.9 * stage_us * (double)longest;
  int64_t best_p = 0;
  for (int64_t rounds = 1; rest > 0 && rounds <= 2; ++rounds) {
    if (pieces(most) > rounds * slots) continue;
    int64_t lo = 0, hi = most;  // the shortest pieces that fit the rounds
    while (hi - lo > 1) {
      const int64_t mid = (lo + hi) / 2;
      (pieces(mid) <= rounds * slots ? hi : lo) = mid;
    }
    const double us = (double)rounds * ((double)hi * stage_us + 2.0) +
                      (double)pieces(hi) * (double)(2 * sizeof(float) * kPieceFloats) / 4e6 + 6.0;
    if (us < best) {
      best = us;
      best_p = hi;
    }
  }
  if (!best_p) {
    for (int e = 0; e < n; ++e) g[e].whole = g[e].tiles;
    return 0;
  }
  for (int e = 0; e < n; ++e)
    if (g[e].tiles > g[e].whole) {
      g[e].pieces_a = (int)((g[e].na + best_p - 1) / best_p);
      g[e].pieces_g = (int)((g[e].ng + best_p - 1) / best_p);
    }
  return pieces(best_p);
}

// The tail groups of the groups order[0, n), and their pieces; split: fp32 rows in three parts.
int64_t launch_tails(const da_factor_side* s1, const da_factor_side* s2, const int64_t* K, const int64_t* D, int64_t es,
                     bool split, const int* order, int n, int64_t slots, TailGroup* g) {
  for (int q = 0; q < n; ++q) {
    const int e = order[q];
    g[q].tiles = ((s1[e].tokens + v2::kBM - 1) / v2::kBM) * ((s2[e].tokens + v2::kBN - 1) / v2::kBN);
    g[q].na = split ? split::kSegs * split::part_elems(K[e]) * 2 / v2::kSB : (K[e] * es + v2::kSB - 1) / v2::kSB;
    g[q].ng = split ? split::kSegs * split::part_elems(D[e]) * 2 / v2::kSB : (D[e] * es + v2::kSB - 1) / v2::kSB;
  }
  return plan_tails(g, n, slots, es == 4 && !split ? 4.0 : 0.95);
}

// Floats of a group's slab slots.
size_t slab_floats(const da_factor_side& s1, const da_factor_side& s2) {
  const int64_t slabs = (s1.tokens + v2::kBM - 1) / v2::kBM * (v2::kBM / kSlab);
  return (size_t)((slabs + s1.batch) * ((s2.tokens + v2::kBN - 1) / v2::kBN + s2.batch));
}

// Groups in order of decreasing reduction length K + D (stable): the tile
// kernel deals tiles to the XCDs round-robin, so this is a longest-first
// schedule on every XCD.  The partial sums land in the same per-pair bins
// whatever the order.
std::vector<int> group_order(int n_groups, const int64_t* K, const int64_t* D) {
  std::vector<int> order(n_groups);
  for (int e = 0; e < n_groups; ++e) order[e] = e;
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return K[x] + D[x] > K[y] + D[y]; });
  return order;
}

// Bytes of a grouped call's split copies (0: it stays on fp32 rows).
size_t split_groups(const da_factor_side* s1, const da_factor_side* s2, int n, const int64_t* K, const int64_t* D,
                    const GroupedPlan& p) {
  const int64_t lim = (1LL << 31) - (1LL << 20);
  int64_t slots = 0;
  if (device_cu_count(&slots) != DA_OK) return 0;
  split::Cost cost;
  size_t bytes = 256;
  for (int e = 0; e < n; ++e) {
    const int64_t ts = split::row_bytes(K[e] > D[e] ? K[e] : D[e]), rows = s1[e].tokens + s2[e].tokens;
    if ((rows + 1) * ts >= lim) return 0;
    for (int64_t r : {s1[e].tokens, s2[e].tokens})
      bytes += split::Builder::bytes(r, K[e]) + split::Builder::bytes(r, D[e]);
    cost.values += (double)rows * (double)(K[e] + D[e]);
    const double tiles = (double)((s1[e].tokens + p.tile_r - 1) / p.tile_r) *
                         (double)((s2[e].tokens + p.tile_c - 1) / p.tile_c);
    cost.tiles(tiles, K[e], 4.0);
    cost.tiles(tiles, D[e], 4.0);
    cost.end_chain();
  }
  return bytes <= split::kMaxBytes && cost.pays(slots) ? bytes : 0;
}

// Layout of the grouped workspace: the partial regions, per group; behind them
// the split copies; behind those the pieces' accumulators and slabs of the
// launch that has most of them.
int grouped_plan(const da_factor_side* s1, const da_factor_side* s2, int n_groups, const int64_t* K,
                 const int64_t* D, int dtype, GroupedPlan* p) {
  if (!valid_dtype(dtype)) return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: bad dtype %d", dtype);
  if (n_groups < 0 || (n_groups > 0 && (!s1 || !s2 || !K || !D)))
    return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: bad group list");
  const int64_t es = (int64_t)elem_bytes(dtype);
  p->part_floats = 0;
  p->split_ws = 0;
  p->tail_ws = 0;
  p->v2 = true;
  for (int e = 0; e < n_groups; ++e) {
    // 32-bit buffer offsets over every group's rows, and both loops non-empty
    const da_factor_side* sd[2] = {&s1[e], &s2[e]};
    for (int q = 0; q < 2; ++q) {
      const int64_t ts = sd[q]->act_tstride > sd[q]->grad_tstride ? sd[q]->act_tstride : sd[q]->grad_tstride;
      const int64_t w = K[e] > D[e] ? K[e] : D[e];
      if (sd[q]->tokens < 0 || ts < 0 || (sd[q]->tokens * ts + w) * es >= (1LL << 31) - (1LL << 20)) p->v2 = false;
    }
    if (D[e] <= 0 || K[e] <= 0) p->v2 = false;
  }
  p->tile_r = p->v2 ? v2::kBM : kBM;
  p->tile_c = p->v2 ? v2::kBN : kBN;
  if (n_groups == 0) { p->ws = 0; return DA_OK; }
  const int64_t b1 = s1[0].batch, b2 = s2[0].batch;
  for (int e = 0; e < n_groups; ++e) {
    if (K[e] < 0 || D[e] < 0) return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: group %d negative width", e);
    if ((K[e] * es) % 16 || (D[e] * es) % 16)
      return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: group %d widths must be multiples of %lld elements",
                       e, (long long)(16 / es));
    if (s1[e].has_bias != s2[e].has_bias)
      return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: group %d sides disagree on has_bias", e);
    const da_factor_side* sides[2] = {&s1[e], &s2[e]};
    for (int q = 0; q < 2; ++q) {
      const da_factor_side* sd = sides[q];
      if (sd->batch != (q ? b2 : b1))
        return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: group %d has a different batch", e);
      if (sd->tokens < 0) return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: negative row count");
      if (sd->batch > 0 && !sd->seg_offsets)
        return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: group %d needs seg_offsets", e);
      if (sd->tokens > 0) {
        if (!sd->act || !sd->grad)
          return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: group %d has a NULL factor", e);
        if (((uintptr_t)sd->act | (uintptr_t)sd->grad) & 15)
          return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: factors must be 16-byte aligned");
        if ((sd->act_tstride * es) % 16 || (sd->grad_tstride * es) % 16)
          return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: row strides must be multiples of 16 bytes");
      }
    }
    const int64_t tr = (s1[e].tokens + p->tile_r - 1) / p->tile_r, tc = (s2[e].tokens + p->tile_c - 1) / p->tile_c;
    p->part_floats += (size_t)((tr + b1) * (tc + b2));
  }
  p->ws = p->part_floats * sizeof(float);
  if (!p->v2) return DA_OK;
  p->ws = align256(p->ws);
  if (dtype == DA_F32) p->split_ws = align256(split_groups(s1, s2, n_groups, K, D, *p));
  int64_t slots = 0;
  if (device_cu_count(&slots) != DA_OK) return DA_OK;  // no device to ask: all tiles run whole
  const std::vector<int> order = group_order(n_groups, K, D);
  for (int g0 = 0; g0 < n_groups; g0 += kMaxGroups) {
    const int n = std::min(n_groups - g0, kMaxGroups);
    TailGroup tails[kMaxGroups];
    const int64_t pieces = launch_tails(s1, s2, K, D, es, p->split_ws > 0, &order[g0], n, slots, tails);
    if (!pieces) continue;
    size_t bytes = (size_t)pieces * kPieceFloats * sizeof(float);
    for (int q = 0; q < n; ++q)
      if (tails[q].whole < tails[q].tiles) bytes += slab_floats(s1[order[g0 + q]], s2[order[g0 + q]]) * sizeof(float);
    p->tail_ws = std::max(p->tail_ws, bytes);
  }
  return DA_OK;
}

// Both entry points: all (i, j) pairs into out[i * ld_out + j], or (diag) the
// pairs (i, i) into out[i * ld_out].
int run_ghost(const da_factor_side* s1, const da_factor_side* s2, int64_t K, int64_t D, int dtype, bool diag,
              float* out, int64_t ld_out, int accumulate, void* workspace, size_t workspace_bytes,
              hipStream_t st) {
  Plan plan;
  int rc = make_plan(s1, s2, K, D, dtype, &plan, diag);
  if (rc) return rc;
  const int64_t b1 = s1->batch, b2 = diag ? 1 : s2->batch;
  if (b1 == 0 || s2->batch == 0) return DA_OK;
  if (!out) return set_error(DA_ERR_INVALID, "da_ghost_gram: out is NULL");
  if (ld_out < b2)
    return set_error(DA_ERR_INVALID, diag ? "da_ghost_gram_diag: out_stride < 1" : "da_ghost_gram: ld_out < B2");
  if (s1->tokens == 0 || s2->tokens == 0) {
    return accumulate ? DA_OK : zero_f32_2d(out, b1, b2, ld_out, st);
  }
  if (!workspace || workspace_bytes < plan.ws)
    return set_error(DA_ERR_WORKSPACE, "da_ghost_gram: workspace needs %zu bytes, got %zu", plan.ws,
                     workspace_bytes);
  const int64_t es = (int64_t)elem_bytes(dtype);
  GhostArgs args;
  args.s1 = to_dev(s1, es);
  args.s2 = to_dev(s2, es);
  args.kbytes_a = K * es;
  args.kbytes_g = D * es;
  args.tiles_r = plan.tiles_r;
  args.tiles_c = plan.tiles_c;
  args.n_r = plan.n_r;
  args.n_c = plan.n_c;
  args.bias = s1->has_bias ? 1.f : 0.f;
  args.diag = diag ? 1 : 0;
  args.partial = (float*)workspace;
  args.gate = Gate{nullptr, 0};
  const int64_t ntiles = plan.n_r * plan.n_c;
  if (ntiles > 0x7fffffffLL) return set_error(DA_ERR_INVALID, "da_ghost_gram: too many tiles");
  dim3 grid((unsigned)ntiles);
  if (plan.split_ws && workspace_bytes >= plan.ws + plan.split_ws) {
    // split fp32 rows on the bf16 pipe; the fp32 launch below runs only for values they cannot hold
    split::Builder b((char*)workspace + plan.ws, st);
    GhostArgs sa = args;
    sa.s1 = split_side(b, args.s1, K, D);
    sa.s2 = split_side(b, args.s2, K, D);
    sa.kbytes_a = split::part_elems(K) * 2;
    sa.kbytes_g = split::part_elems(D) * 2;
    rc = b.flush();
    if (rc) return rc;
    sa.gate = Gate{b.flag(), 0};
    args.gate = Gate{b.flag(), 1};
    ghost_gram_tiles_v3<DA_BF16, 3><<<grid, v3::kThreads, 0, st>>>(sa);
    rc = check_launch("da_ghost_gram(split tiles)");
    if (rc) return rc;
  }
  if (plan.v2) {
    switch (dtype) {
      case DA_BF16: ghost_gram_tiles_v3<DA_BF16><<<grid, v3::kThreads, 0, st>>>(args); break;
      case DA_F16: ghost_gram_tiles_v3<DA_F16><<<grid, v3::kThreads, 0, st>>>(args); break;
      default: ghost_gram_tiles_v3<DA_F32><<<grid, v3::kThreads, 0, st>>>(args); break;
    }
  } else {
    switch (dtype) {
      case DA_BF16: ghost_gram_tiles<DA_BF16><<<grid, kThreads, 0, st>>>(args); break;
      case DA_F16: ghost_gram_tiles<DA_F16><<<grid, kThreads, 0, st>>>(args); break;
      default: ghost_gram_tiles<DA_F32><<<grid, kThreads, 0, st>>>(args); break;
    }
  }
  rc = check_launch("da_ghost_gram(tiles)");
  if (rc) return rc;
  const int64_t pairs = b1 * b2;
  ghost_gram_reduce<<<(unsigned)((pairs + 255) / 256), 256, 0, st>>>(
      (const float*)workspace, b1, b2, plan.per_pair, out, ld_out, accumulate);
  return check_launch("da_ghost_gram(reduce)");
}

}  // namespace
}  // namespace da

extern "C" {

int da_ghost_gram_workspace(const da_factor_side* s1, const da_factor_side* s2, int64_t K,
                            int64_t D, int dtype, size_t* bytes) {
  da::Plan plan;
  int rc = da::make_plan(s1, s2, K, D, dtype, &plan);
  if (rc) return rc;
  if (!bytes) return da::set_error(DA_ERR_INVALID, "da_ghost_gram_workspace: bytes is NULL");
  *bytes = plan.ws + plan.split_ws;
  return DA_OK;
}

int da_ghost_gram_workspace_min(const da_factor_side* s1, const da_factor_side* s2, int64_t K, int64_t D, int dtype,
                                int diag, size_t* bytes) {
  da::Plan plan;
  int rc = da::make_plan(s1, s2, K, D, dtype, &plan, diag != 0);
  if (rc) return rc;
  if (!bytes) return da::set_error(DA_ERR_INVALID, "da_ghost_gram_workspace_min: bytes is NULL");
  *bytes = plan.ws;
  return DA_OK;
}

int da_ghost_gram(const da_factor_side* s1, const da_factor_side* s2, int64_t K, int64_t D,
                  int dtype, float* out, int64_t ld_out, int accumulate, void* workspace,
                  size_t workspace_bytes, void* stream) {
  return da::run_ghost(s1, s2, K, D, dtype, false, out, ld_out, accumulate, workspace, workspace_bytes,
                       (hipStream_t)stream);
}

int da_ghost_gram_diag_workspace(const da_factor_side* s1, const da_factor_side* s2, int64_t K, int64_t D,
                                 int dtype, size_t* bytes) {
  da::Plan plan;
  int rc = da::make_plan(s1, s2, K, D, dtype, &plan, true);
  if (rc) return rc;
  if (!bytes) return da::set_error(DA_ERR_INVALID, "da_ghost_gram_diag_workspace: bytes is NULL");
  *bytes = plan.ws + plan.split_ws;
  return DA_OK;
}

int da_ghost_gram_diag(const da_factor_side* s1, const da_factor_side* s2, int64_t K, int64_t D, int dtype,
                       float* out, int64_t out_stride, int accumulate, void* workspace, size_t workspace_bytes,
                       void* stream) {
  return da::run_ghost(s1, s2, K, D, dtype, true, out, out_stride, accumulate, workspace, workspace_bytes,
                       (hipStream_t)stream);
}

int da_ghost_gram_grouped_workspace(const da_factor_side* s1, const da_factor_side* s2, int n_groups,
                                    const int64_t* K, const int64_t* D, int dtype, size_t* bytes) {
  da::GroupedPlan plan;
  int rc = da::grouped_plan(s1, s2, n_groups, K, D, dtype, &plan);
  if (rc) return rc;
  if (!bytes) return da::set_error(DA_ERR_INVALID, "da_ghost_gram_grouped_workspace: bytes is NULL");
  *bytes = plan.ws + plan.split_ws + plan.tail_ws;
  return DA_OK;
}

int da_ghost_gram_grouped_workspace_min(const da_factor_side* s1, const da_factor_side* s2, int n_groups,
                                        const int64_t* K, const int64_t* D, int dtype, size_t* bytes) {
  da::GroupedPlan plan;
  int rc = da::grouped_plan(s1, s2, n_groups, K, D, dtype, &plan);
  if (rc) return rc;
  if (!bytes) return da::set_error(DA_ERR_INVALID, "da_ghost_gram_grouped_workspace_min: bytes is NULL");
  *bytes = plan.ws;
  return DA_OK;
}

int da_ghost_gram_grouped(const da_factor_side* s1, const da_factor_side* s2, int n_groups,
                          const int64_t* K, const int64_t* D, int dtype, float* out, int64_t ld_out,
                          int accumulate, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace da;
  GroupedPlan plan;
  int rc = grouped_plan(s1, s2, n_groups, K, D, dtype, &plan);
  if (rc) return rc;
  if (n_groups == 0) return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: no groups");
  const int64_t b1 = s1[0].batch, b2 = s2[0].batch;
  if (b1 == 0 || b2 == 0) return DA_OK;
  if (!out) return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: out is NULL");
  if (ld_out < b2) return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: ld_out < B2");
  if (!workspace || workspace_bytes < plan.ws)
    return set_error(DA_ERR_WORKSPACE, "da_ghost_gram_grouped: workspace needs %zu bytes, got %zu", plan.ws,
                     workspace_bytes);
  hipStream_t st = (hipStream_t)stream;
  const int64_t es = (int64_t)elem_bytes(dtype);
  float* part = (float*)workspace;
  int64_t part_off = 0;
  bool first_launch = true;
  const bool split_rows = plan.split_ws && workspace_bytes >= plan.ws + plan.split_ws;
  split::Builder copies(split_rows ? (char*)workspace + plan.ws : nullptr, st);
  // With less memory than the query asked for, all tiles run whole.
  const bool pieces_fit = plan.tail_ws && workspace_bytes >= plan.ws + plan.split_ws + plan.tail_ws;
  float* const dump = pieces_fit ? (float*)((char*)workspace + plan.ws + plan.split_ws) : nullptr;
  int64_t slots = 0;
  if (pieces_fit && (rc = device_cu_count(&slots)) != DA_OK) return rc;
  const std::vector<int> order = group_order(n_groups, K, D);
  for (int g0 = 0; g0 < n_groups; g0 += kMaxGroups) {
    const int n = n_groups - g0 < kMaxGroups ? n_groups - g0 : kMaxGroups;
    GroupedArgs ga;
    ga.n_groups = 0;
    ga.tile_r = plan.tile_r;
    ga.tile_c = plan.tile_c;
    ga.b1 = b1;
    ga.b2 = b2;
    ga.partial = part;
    ga.dump = dump;
    ga.gate = Gate{nullptr, 0};
    TailGroup tails[kMaxGroups];
    const int64_t pieces =
        pieces_fit ? launch_tails(s1, s2, K, D, es, split_rows, &order[g0], n, slots, tails) : 0;
    int64_t tiles = 0, whole = 0, piece0 = 0;
    int64_t slab_off = pieces ? dump - part + pieces * kPieceFloats : 0;
    for (int q = 0; q < n; ++q) {
      const int e = order[g0 + q];
      const da_factor_side& x = s1[e];
      const da_factor_side& y = s2[e];
      const int64_t tr = (x.tokens + plan.tile_r - 1) / plan.tile_r, tc = (y.tokens + plan.tile_c - 1) / plan.tile_c;
      GroupDev& G = ga.grp[ga.n_groups++];
      G.a1 = (const char*)x.act;
      G.g1 = (const char*)x.grad;
      G.a2 = (const char*)y.act;
      G.g2 = (const char*)y.grad;
      G.seg1 = x.seg_offsets;
      G.seg2 = y.seg_offsets;
      G.idx1 = x.row_index;
      G.idx2 = y.row_index;
      G.rows1 = x.tokens;
      G.rows2 = y.tokens;
      G.a1_ts = x.act_tstride * es;
      G.g1_ts = x.grad_tstride * es;
      G.a2_ts = y.act_tstride * es;
      G.g2_ts = y.grad_tstride * es;
      if (tiles + tr * tc > 0x7fffffffLL) return set_error(DA_ERR_INVALID, "da_ghost_gram_grouped: too many tiles");
      G.tile0 = (int32_t)whole;
      G.piece0 = (int32_t)piece0;
      G.tiles_r = (int32_t)tr;
      G.tiles_c = (int32_t)tc;
      G.whole = (int32_t)(pieces ? tails[q].whole : tr * tc);
      G.pieces_a = (int16_t)(pieces ? tails[q].pieces_a : 0);
      G.pieces_g = (int16_t)(pieces ? tails[q].pieces_g : 0);
      G.part_off = part_off;
      G.part_ld = tc + b2;
      G.slab_off = slab_off;
      G.kbytes_a = K[e] * es;
      G.kbytes_g = D[e] * es;
      G.bias = x.has_bias ? 1.f : 0.f;
      tiles += tr * tc;
      whole += G.whole;
      piece0 += (tr * tc - G.whole) * (G.pieces_a + G.pieces_g);
      if (G.whole < tr * tc) slab_off += (int64_t)slab_floats(x, y);
      part_off += (tr + b1) * (tc + b2);
    }
    ga.whole = (int)whole;
    const unsigned grid = (unsigned)(whole + pieces), finish = (unsigned)((tiles - whole) * (v2::kBM / kSlab));
    GroupedArgs reduce = ga;  // where the sums of a pair lie
    if (tiles > 0) {
      if (split_rows) {
        // Live rows split in packed order on the bf16 pipe; the fp32 launch
        // below runs only for values they cannot hold (one flag for the call:
        // a later launch's values may raise it too, never clear it).
        GroupedArgs sa = ga;
        for (int q = 0; q < n; ++q) {
          const int e = order[g0 + q];
          GroupDev& G = sa.grp[q];
          const int32_t* live1 = G.seg1 + b1;
          const int32_t* live2 = G.seg2 + b2;
          G.a1 = copies.add(G.a1, 1, G.rows1, 0, G.a1_ts, K[e], G.idx1, live1);
          G.g1 = copies.add(G.g1, 1, G.rows1, 0, G.g1_ts, D[e], G.idx1, live1);
          G.a2 = copies.add(G.a2, 1, G.rows2, 0, G.a2_ts, K[e], G.idx2, live2);
          G.g2 = copies.add(G.g2, 1, G.rows2, 0, G.g2_ts, D[e], G.idx2, live2);
          G.idx1 = G.idx2 = nullptr;
          G.a1_ts = G.a2_ts = split::row_bytes(K[e]);
          G.g1_ts = G.g2_ts = split::row_bytes(D[e]);
          G.kbytes_a = split::part_elems(K[e]) * 2;
          G.kbytes_g = split::part_elems(D[e]) * 2;
        }
        rc = copies.flush();
        if (rc) return rc;
        reduce.gate = sa.gate = Gate{copies.flag(), 0};
        ga.gate = Gate{copies.flag(), 1};
        ghost_grouped_tiles_v3<DA_BF16, 3><<<grid, v3::kThreads, 0, st>>>(sa);
        rc = check_launch("da_ghost_gram_grouped(split tiles)");
        if (rc) return rc;
        if (finish) {
          ghost_grouped_finish<<<finish, kFinishThreads, 0, st>>>(sa);
          rc = check_launch("da_ghost_gram_grouped(split finish)");
          if (rc) return rc;
        }
        // the fp32 launch takes every tile whole
        whole = 0;
        for (int q = 0; q < ga.n_groups; ++q) {
          GroupDev& G = ga.grp[q];
          G.whole = G.tiles_r * G.tiles_c;
          G.tile0 = (int32_t)whole;
          whole += G.whole;
        }
        ga.whole = (int)whole;
      }
      if (plan.v2) {
        const unsigned blocks = split_rows ? (unsigned)tiles : grid;
        switch (dtype) {
          case DA_BF16: ghost_grouped_tiles_v3<DA_BF16><<<blocks, v3::kThreads, 0, st>>>(ga); break;
          case DA_F16: ghost_grouped_tiles_v3<DA_F16><<<blocks, v3::kThreads, 0, st>>>(ga); break;
          default: ghost_grouped_tiles_v3<DA_F32><<<blocks, v3::kThreads, 0, st>>>(ga); break;
        }
        if (finish && !split_rows) {
          rc = check_launch("da_ghost_gram_grouped(tiles)");
          if (rc) return rc;
          ghost_grouped_finish<<<finish, kFinishThreads, 0, st>>>(ga);
        }
      } else {
        switch (dtype) {
          case DA_BF16: ghost_grouped_tiles<DA_BF16><<<(unsigned)tiles, kThreads, 0, st>>>(ga); break;
          case DA_F16: ghost_grouped_tiles<DA_F16><<<(unsigned)tiles, kThreads, 0, st>>>(ga); break;
          default: ghost_grouped_tiles<DA_F32><<<(unsigned)tiles, kThreads, 0, st>>>(ga); break;
        }
      }
      rc = check_launch("da_ghost_gram_grouped(tiles)");
      if (rc) return rc;
    }
    grouped_reduce<<<(unsigned)((b1 * b2 + 3) / 4), 256, 0, st>>>(reduce, out, ld_out,
                                                                    (accumulate || !first_launch) ? 1 : 0);
    rc = check_launch("da_ghost_gram_grouped(reduce)");
    if (rc) return rc;
    first_launch = false;
  }
  return DA_OK;
}


int da_ghost_gram_per_token_workspace(const da_factor_side* s1, const da_factor_side* s2, int64_t K, int64_t D,
                                      int dtype, size_t* bytes) {
  using namespace da;
  if (!bytes || !s2) return set_error(DA_ERR_INVALID, "da_ghost_gram_per_token_workspace: NULL argument");
  PerTokPlan p;
  const int rc = per_token_plan(s1, s2->batch, s2->tokens, K, D, dtype, "da_ghost_gram_per_token", &p);
  if (rc) return rc;
  per_token_split(s1, s2, K, D, dtype, &p);
  *bytes = p.ws + p.split_ws;
  return DA_OK;
}

int da_ghost_gram_per_token_workspace_min(const da_factor_side* s1, const da_factor_side* s2, int64_t K, int64_t D,
                                          int dtype, size_t* bytes) {
  using namespace da;
  if (!bytes || !s2) return set_error(DA_ERR_INVALID, "da_ghost_gram_per_token_workspace_min: NULL argument");
  PerTokPlan p;
  const int rc = per_token_plan(s1, s2->batch, s2->tokens, K, D, dtype, "da_ghost_gram_per_token", &p);
  if (rc) return rc;
  per_token_split(s1, s2, K, D, dtype, &p);
  *bytes = p.ws;
  return DA_OK;
}

int da_ghost_gram_per_token(const da_factor_side* s1, const da_factor_side* s2, int64_t K, int64_t D, int dtype,
                            float* out, int64_t ld_b1, int64_t ld_t, int64_t ld_b2, int accumulate,
                            void* workspace, size_t workspace_bytes, void* stream) {
  using namespace da;
  const char* who = "da_ghost_gram_per_token";
  if (!s1 || !s2) return set_error(DA_ERR_INVALID, "%s: NULL side", who);
  PerTokPlan p;
  int rc = per_token_plan(s1, s2->batch, s2->tokens, K, D, dtype, who, &p);
  if (rc) return rc;
  rc = validate_side(s1, K, D, dtype, "s1");
  if (rc) return rc;
  rc = validate_side(s2, K, D, dtype, "s2");
  if (rc) return rc;
  if (s1->has_bias != s2->has_bias) return set_error(DA_ERR_INVALID, "%s: both sides must agree on has_bias", who);
  if (s1->batch == 0 || s1->tokens == 0 || s2->batch == 0) return DA_OK;
  if (!out) return set_error(DA_ERR_INVALID, "%s: out is NULL", who);
  const int64_t es = (int64_t)elem_bytes(dtype);
  if (s1->seg_offsets || s2->seg_offsets || !fits_v2(s1, K, D, es) || !fits_v2(s2, K, D, es) || D == 0 || K == 0)
    return set_error(DA_ERR_UNSUPPORTED,
                     "%s: needs dense sides with rows addressable by 32-bit offsets, K > 0 and D > 0", who);
  per_token_split(s1, s2, K, D, dtype, &p);
  if (!workspace || workspace_bytes < p.ws)
    return set_error(DA_ERR_WORKSPACE, "%s: workspace needs %zu bytes", who, p.ws);
  PerTokArgs g;
  g.gate = Gate{nullptr, 0};
  g.s1 = to_dev(s1, es);
  g.s2 = to_dev(s2, es);
  g.kbytes_a = K * es;
  g.kbytes_g = D * es;
  g.tiles_r = p.tiles_r;
  g.tiles_c = p.tiles_c;
  g.n_r = s1->batch * p.tiles_r;
  g.n_c = s2->batch * p.tiles_c;
  g.bias = s1->has_bias ? 1.f : 0.f;
  g.m2bias = nullptr;
  g.m2bias_ld = 0;
  g.tpad = p.tpad;
  g.partial = (float*)workspace;
  if (s2->tokens == 0) {  // nothing on side 2: the sums are zero
    g.tiles_c = 0;
    const int64_t n = s1->batch * s1->tokens * s2->batch;
    per_token_reduce<<<(unsigned)((n + 255) / 256), 256, 0, (hipStream_t)stream>>>(
        g.partial, s1->batch, s1->tokens, s2->batch, g.tpad, 0, out, ld_b1, ld_t, ld_b2, accumulate);
    return check_launch(who);
  }
  if (p.split_ws && workspace_bytes >= p.ws + p.split_ws) {
    split::Builder b((char*)workspace + p.ws, (hipStream_t)stream);
    PerTokArgs sa = g;
    sa.s1 = split_side(b, g.s1, K, D);
    sa.s2 = split_side(b, g.s2, K, D);
    sa.kbytes_a = split::part_elems(K) * 2;
    sa.kbytes_g = split::part_elems(D) * 2;
    rc = b.flush();
    if (rc) return rc;
    sa.gate = Gate{b.flag(), 0};
    g.gate = Gate{b.flag(), 1};
    const int64_t tiles = g.n_r * g.n_c;
    if (tiles > 0x7fffffffLL) return set_error(DA_ERR_INVALID, "%s: problem too large", who);
    ghost_per_token_v3<DA_BF16, false, 3><<<(unsigned)tiles, v3::kThreads, 0, (hipStream_t)stream>>>(sa);
    rc = check_launch(who);
    if (rc) return rc;
  }
  return per_token_launch(g, false, dtype, s1->tokens, out, ld_b1, ld_t, ld_b2, accumulate, (hipStream_t)stream, who);
}

int da_dense_per_token_workspace(const da_factor_side* s1, int64_t b2, int64_t K, int64_t D, int dtype,
                                 size_t* bytes) {
  using namespace da;
  if (!bytes) return set_error(DA_ERR_INVALID, "da_dense_per_token_workspace: bytes is NULL");
  PerTokPlan p;
  const int rc = per_token_plan(s1, b2, D, K, D, dtype, "da_dense_per_token", &p);
  if (rc) return rc;
  *bytes = p.ws;
  return DA_OK;
}

int da_dense_per_token(const da_factor_side* s1, const void* m2, int64_t b2, int64_t m2_bstride, int64_t m2_rstride,
                       const float* m2_bias, int64_t m2_bias_ld, int64_t K, int64_t D, int dtype, float* out,
                       int64_t ld_b1, int64_t ld_t, int64_t ld_b2, int accumulate, void* workspace,
                       size_t workspace_bytes, void* stream) {
  using namespace da;
  const char* who = "da_dense_per_token";
  PerTokPlan p;
  int rc = per_token_plan(s1, b2, D, K, D, dtype, who, &p);
  if (rc) return rc;
  rc = validate_side(s1, K, D, dtype, "s1");
  if (rc) return rc;
  if (s1->batch == 0 || s1->tokens == 0 || b2 == 0) return DA_OK;
  if (!out) return set_error(DA_ERR_INVALID, "%s: out is NULL", who);
  const int64_t es = (int64_t)elem_bytes(dtype);
  if (K == 0 || D == 0) return set_error(DA_ERR_UNSUPPORTED, "%s: needs K > 0 and D > 0", who);
  if (!m2 || ((uintptr_t)m2 & 15) || (m2_bstride * es) % 16 || (m2_rstride * es) % 16 || m2_rstride < K ||
      m2_bstride < 0)
    return set_error(DA_ERR_INVALID, "%s: m2 rows must be 16-byte aligned, row stride >= K", who);
  if (s1->has_bias && !m2_bias) return set_error(DA_ERR_INVALID, "%s: a bias column needs m2_bias", who);
  const int64_t lim = (1LL << 31) - (1LL << 20);
  if (s1->seg_offsets || !fits_v2(s1, K, D, es) || D * m2_rstride * es + K * es >= lim)
    return set_error(DA_ERR_UNSUPPORTED, "%s: needs a dense side 1 and rows addressable by 32-bit offsets", who);
  if (!workspace || workspace_bytes < p.ws)
    return set_error(DA_ERR_WORKSPACE, "%s: workspace needs %zu bytes", who, p.ws);
  PerTokArgs g;
  g.gate = Gate{nullptr, 0};
  g.s1 = to_dev(s1, es);
  g.s2.act = (const char*)m2;
  g.s2.grad = (const char*)m2;
  g.s2.batch = b2;
  g.s2.tokens = D;  // M2_j's rows (output channels) take side 2's tokens
  g.s2.act_bstride = g.s2.grad_bstride = m2_bstride * es;
  g.s2.act_tstride = g.s2.grad_tstride = m2_rstride * es;
  g.s2.seg = nullptr;
  g.s2.idx = nullptr;
  g.kbytes_a = 0;  // one product: a1 rows against M2_j rows over K
  g.kbytes_g = K * es;
  g.tiles_r = p.tiles_r;
  g.tiles_c = p.tiles_c;
  g.n_r = s1->batch * p.tiles_r;
  g.n_c = b2 * p.tiles_c;
  g.bias = 0.f;
  g.m2bias = s1->has_bias ? m2_bias : nullptr;
  g.m2bias_ld = m2_bias_ld;
  g.tpad = p.tpad;
  g.partial = (float*)workspace;
  return per_token_launch(g, true, dtype, s1->tokens, out, ld_b1, ld_t, ld_b2, accumulate, (hipStream_t)stream, who);
}

}  // extern "C"
