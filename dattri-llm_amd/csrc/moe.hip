// K3c: MoE routing and expert segmentation (integer work, bit-exact).
//
//   da_moe_topk:       top-k of softmax(logits) per token, weights renormalised
//                      over the k, indices in torch.topk's CPU order (ties
//                      included, topk_select.h) -- the router of
//                      transformers' MixtralTopKRouter.forward
//                      (softmax(logits.float()) -> topk -> / sum), as consumed by
//                      dattri_llm/gradient/hooks/override_layers/fused_experts.py:210-237.
//   da_counting_sort:  stable counting sort of int32 keys into bins.  With the
//                      top-k indices read slot-major (key[p] = idx[p % N][p / N])
//                      the sorted order is exactly the reference loop's
//                      torch.where(one_hot(idx).permute(2,1,0)[e]) enumeration,
//                      fused_experts.py:219-228 (slot-major, token ascending),
//                      and the bin offsets are the expert segments.  With
//                      key = token // T it groups an expert's rows by sample for
//                      the segmented ghost product (the dense-with-zeros regroup
//                      of hooks/routing.py:71-86, without the zeros).
//
// Both are tiny next to the expert GEMMs; they exist so the routing never
// leaves the device and never depends on a library sort's tie order.
#include <atomic>

#include "common.h"
#include "topk_select.h"

namespace da {
namespace {

constexpr int kMaxExperts = 256;
constexpr int kMaxTopK = 16;
constexpr int kMaxBins = 8192;

// One router queue per lane in LDS: entry i of lane l at [i * lanes + l], so
// the lanes of a wave touching the same entry hit consecutive words.
struct LdsQueue {
  float* p;
  uint16_t* e;
  int lanes;
  __device__ topk::Entry get(int i) const { return {p[i * lanes], (int)e[i * lanes]}; }
  __device__ void set(int i, topk::Entry x) {
    p[i * lanes] = x.p;
    e[i * lanes] = (uint16_t)x.e;
  }
  __device__ void swap(int i, int j) {
    const topk::Entry a = get(i), b = get(j);
    set(i, b);
    set(j, a);
  }
};

// One lane per token (workgroups of 64 lanes, 32 above 128 experts, so the
// dynamic LDS of 6 bytes per expert and 4 per slot of a lane stays within 52
// KB).  softmax(logits.float()) as torch computes it -- a maximum that
// propagates NaN, then exp(x - max) / sum -- so a row holding a NaN or +inf
// logit, or only -inf logits, gives NaN probabilities as torch's does; then
// the selection and weights = top / sum(top).
// Where no two of the k largest probabilities are equal their order is the only
// one any selection can give, and k passes for the largest value below the last
// find it without a branch; other lanes (ties, NaN) run the selection of
// topk_select.h, whose lanes part ways at every comparison.  4096 tokens, 64
// experts, top-8: 134 us by that selection alone, 30 by the passes (bf16 logits,
// with ties in most waves: 138 and 125).  Above 128 experts a wave with a tie
// gives up the passes, and 16-bit logits, which nearly always have one, skip
// them (256 experts, top-16: 493 us, 639 with all passes first; fp32 486 and 225).
// Up to 128 the lanes without a tie still gain, until bf16 has too many: 64
// experts, bf16, top-8 117 us with the passes and 151 without, top-12 148 and 160,
// top-16 177 and 160 (128 experts 360 and 300); fp16 top-16 140 and 182.
template <int DT>
__global__ __launch_bounds__(kWave) void moe_topk_kernel(const char* logits, int64_t n, int e, int k,
                                                         int64_t rstride, float* weights, int64_t* index) {
  extern __shared__ __attribute__((aligned(16))) char topk_lds[];
  const int lane = threadIdx.x, lanes = blockDim.x;
  const int64_t tok = (int64_t)blockIdx.x * lanes + lane;
  if (tok >= n) return;
  LdsQueue q{(float*)topk_lds + lane, (uint16_t*)(topk_lds + (size_t)e * lanes * 4) + lane, lanes};
  const char* row = logits + tok * rstride * Elem<DT>::kBytes;
  float mx = -INFINITY;
#pragma unroll 8
  for (int x = 0; x < e; ++x) {
    const float v = Elem<DT>::load(row, x);
    q.p[x * lanes] = v;
    if (mx == mx && (v != v || v > mx)) mx = v;
  }
  float sum = 0.f;
  for (int x = 0; x < e; ++x) {
    const float v = expf(q.p[x * lanes] - mx);
    q.p[x * lanes] = v;
    sum += v;
  }
  for (int x = 0; x < e; ++x) q.set(x, {q.p[x * lanes] / sum, x});
  float* const top = (float*)(topk_lds + (size_t)e * lanes * 6) + lane;
  float below = INFINITY, tsum = 0.f;
  const bool many = lanes < kWave;  // above 128 experts
  const bool skip = (many && Elem<DT>::kBytes == 2) || (DT == DA_BF16 && k > 12);
  bool unique = !skip;
  for (int s = 0; s < k && !skip && !(many && __any(!unique)); ++s) {
    float m = -1.f;
    int at = 0, equal = 0;
#pragma unroll 8
    for (int x = 0; x < e; ++x) {
      const float v = q.p[x * lanes];
      const bool in = v < below, up = in & (v > m);
      equal = up ? 1 : equal + (int)(in & (v == m));
      at = up ? x : at;
      m = up ? v : m;
    }
    unique &= equal == 1;
    below = m;
    top[s * lanes] = m;
    tsum += m;
    index[tok * k + s] = at;
  }
  if (many && __any(!unique)) unique = false;  // the wave's passes may not have ended
  if (unique) {
    for (int s = 0; s < k; ++s) weights[tok * k + s] = top[s * lanes] / tsum;
    return;
  }
  topk::select_topk(q, e, k);
  tsum = 0.f;
  for (int s = 0; s < k; ++s) tsum += q.get(s).p;
  for (int s = 0; s < k; ++s) {
    const topk::Entry t = q.get(s);
    weights[tok * k + s] = t.p / tsum;
    index[tok * k + s] = t.e;
  }
}

// Routed-row compaction: the rows p < batch * tokens whose mask byte is
// non-zero, in increasing order, with per-sample offsets (row p = b * tokens
// + t belongs to sample b).  One workgroup, bound by the latency of its steps:
// a thread takes 16 consecutive mask bytes (one load), so a step is 16384
// rows, ranked by a scan of the threads' counts and a running carry (a byte per
// thread: 17 us for 16384 rows and 33 for 32768; now 9 and 14).
constexpr int kCompactBytes = 16;
__global__ __launch_bounds__(1024) void compact_rows_kernel(const uint8_t* __restrict__ mask, int64_t batch,
                                                            int64_t tokens, int32_t* __restrict__ seg,
                                                            int32_t* __restrict__ rows) {
  __shared__ int32_t wave_count[2][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t n = batch * tokens;
  if (tokens == 0)
    for (int64_t b = tid; b < batch; b += 1024) seg[b] = 0;  // no rows to write them from
  const bool aligned = ((uintptr_t)mask & 15) == 0;
  int32_t carry = 0;
  int buf = 0;
  for (int64_t base = 0; base < n; base += 1024 * kCompactBytes, buf ^= 1) {
    const int64_t p0 = base + tid * kCompactBytes;
    const int live = (int)max((int64_t)0, min((int64_t)kCompactBytes, n - p0));
    uint32_t word[4] = {0, 0, 0, 0};
    if (aligned && live == kCompactBytes) {
      const u32x4 v = ld16((const char*)mask + p0);
#pragma unroll
      for (int j = 0; j < 4; ++j) word[j] = v[j];
    } else {
#pragma unroll
      for (int j = 0; j < kCompactBytes; ++j)
        if (j < live) word[j >> 2] |= (uint32_t)mask[p0 + j] << (8 * (j & 3));
    }
    uint32_t keep = 0;
#pragma unroll
    for (int j = 0; j < kCompactBytes; ++j) keep |= (uint32_t)(((word[j >> 2] >> (8 * (j & 3))) & 0xffu) != 0) << j;
    const int32_t mine = __popc(keep);
    int32_t upto = mine;  // inclusive over the wave
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int32_t y = __shfl_up(upto, off, 64);
      if (lane >= off) upto += y;
    }
    if (lane == 63) wave_count[buf][wave] = upto;
    // one barrier a step: the next step writes the other buffer, and the one after
    // that is behind the next step's barrier
    __syncthreads();
    int32_t rank = carry + upto - mine;  // kept rows before p0
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const int32_t c = wave_count[buf][w];
      if (w < wave) rank += c;
      carry += c;
    }
    if (live > 0) {
      int64_t b = (p0 + tokens - 1) / tokens, start = b * tokens;  // the first sample that starts here or later
#pragma unroll
      for (int j = 0; j < kCompactBytes; ++j) {
        if (j >= live) break;
        if (p0 + j == start) {
          seg[b++] = rank;
          start += tokens;
        }
        if (keep >> j & 1) rows[rank++] = (int32_t)(p0 + j);
      }
    }
  }
  if (tid == 0) seg[batch] = carry;
}

// keys are read either directly (slot_major == 0: key[p] = keys[p]) or as the
// slot-major view of an (n/k, k) int64 index matrix (slot_major == 1).
struct SortArgs {
  const int32_t* keys32;
  const int64_t* keys64;  // (rows, k) row-major when slot_major
  int64_t n, rows, k;
  int slot_major;
  int bins;
  int32_t* offsets;       // bins + 1
  int32_t* perm;          // n
  int64_t key_div;        // key = raw / key_div (1 = identity)
};

__device__ __forceinline__ int64_t sort_key(const SortArgs& a, int64_t p) {
  int64_t raw;
  if (a.slot_major) {
    const int64_t slot = p / a.rows, r = p - slot * a.rows;
    raw = a.keys64[r * a.k + slot];
  } else {
    raw = a.keys32 ? (int64_t)a.keys32[p] : a.keys64[p];
  }
  return a.key_div > 1 ? (raw >= 0 ? raw / a.key_div : -1) : raw;
}

// One workgroup: histogram (LDS atomics; counts are order independent), exclusive
// scan, then wave 0 scatters in input order, 64 entries at a time, ranking equal
// keys inside the wave with shuffles -- a stable sort.  Keys outside [0, bins)
// are skipped; offsets[bins] is the number of entries kept.
__global__ __launch_bounds__(256) void counting_sort_kernel(SortArgs a) {
  __shared__ int32_t cnt[kMaxBins];
  const int tid = threadIdx.x;
  for (int b = tid; b < a.bins; b += 256) cnt[b] = 0;
  __syncthreads();
  for (int64_t p = tid; p < a.n; p += 256) {
    const int64_t key = sort_key(a, p);
    if (key >= 0 && key < a.bins) atomicAdd(&cnt[key], 1);
  }
  __syncthreads();
  if (tid == 0) {
    int32_t run = 0;
    for (int b = 0; b < a.bins; ++b) {
      const int32_t c = cnt[b];
      a.offsets[b] = run;
      cnt[b] = run;  // becomes the next free slot of bin b
      run += c;
    }
    a.offsets[a.bins] = run;
  }
  __syncthreads();
  if (tid >= 64) return;
  const int lane = tid;
  for (int64_t base = 0; base < a.n; base += 64) {
    const int64_t p = base + lane;
    const int64_t key = p < a.n ? sort_key(a, p) : -1;
    const bool ok = key >= 0 && key < a.bins;
    int rank = 0, total = 0;
    for (int src = 0; src < 64; ++src) {
      const int64_t other = __shfl(key, src, 64);
      if (ok && other == key) {
        total += 1;
        if (src < lane) rank += 1;
      }
    }
    int32_t slot = 0;
    if (ok) slot = cnt[key] + rank;
    // every lane has read cnt[] before the last lane of each key group bumps it
    __builtin_amdgcn_wave_barrier();
    if (ok) {
      a.perm[slot] = (int32_t)p;
      if (rank == total - 1) cnt[key] = slot + 1;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// Expert routing of one side.  Entries p = slot*N + token are visited in order
// (the reference's slot-major enumeration); with e = idx[token][slot] and b =
// token / T two stable sorts come out:
//   by e      -> entries[off[e] + r] = p for expert e's local row r (routed order);
//   by (e, b) -> rows[off[e] + seg[e][b] + q] = r, expert e's local rows grouped by sample,
// with seg[e*(B+1) + b] the start of sample b among expert e's rows.
// A workgroup takes one expert and walks all entries twice: the routing is
// bound by latency, not by the 8 bytes an entry has, and every expert's order
// is then a matter of ballots and running counts, with no sort.  The first walk
// counts the entries of lower experts (off[e]) and leaves the rank R[f] of the
// first position of every (slot, sample) block f = p / T, T consecutive
// entries.  Sample b holds the blocks f = b mod B, so its rows are the differences of
// R summed over the slots, and an entry of rank r in block f goes to place
// D[f] + r of its expert's rows, D formed from R once.  The second walk writes.
// One workgroup that sorted all entries took 31 us for 4096 tokens, 8 experts,
// top-2, and 667 us for 16384 tokens, 64 experts, top-8; now 14 and 111.
struct RouteArgs {
  const int64_t* index;  // (N, k)
  int64_t n, k, experts, batch, tokens;
  int32_t* offsets;  // experts + 1
  int32_t* entries;  // n*k
  int32_t* seg;      // experts * (batch + 1)
  int32_t* rows;     // n*k
};

constexpr int kRouteThreads = 1024;
constexpr int kRouteWaves = kRouteThreads / 64;
constexpr int kRouteRun = 8;           // entries per thread and step
// (slot, sample) blocks whose R and D fit LDS: all of them for k <= experts, as
// every router has it, with at most kMaxBins (expert, sample) pairs.
constexpr int64_t kRouteBlocks = kMaxBins;
inline size_t route_lds(int64_t blocks, int64_t batch) { return (size_t)(2 * blocks + 1 + batch) * sizeof(int32_t); }

// In-place exclusive scan of the LDS array a[0, len) by the whole workgroup.
__device__ void route_scan(int32_t* a, int len, int32_t* wsum) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int per = (len + kRouteThreads - 1) / kRouteThreads;
  const int beg = tid * per;
  int32_t s = 0;
  for (int i = 0; i < per; ++i)
    if (beg + i < len) s += a[beg + i];
  int32_t x = s;  // inclusive scan over the wave
  for (int off = 1; off < 64; off <<= 1) {
    const int32_t y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) wsum[wave] = x;
  __syncthreads();
  int32_t run = x - s;
  for (int w = 0; w < wave; ++w) run += wsum[w];
  for (int i = 0; i < per; ++i)
    if (beg + i < len) {
      const int32_t c = a[beg + i];
      a[beg + i] = run;
      run += c;
    }
  __syncthreads();
}

__global__ __launch_bounds__(kRouteThreads) void moe_route_kernel(RouteArgs a) {
  extern __shared__ int32_t route_mem[];  // R (blocks + 1), D (blocks), seg (B)
  __shared__ int32_t count[2][kRouteWaves], wsum[kRouteWaves];
  __shared__ int32_t lower, valid;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t n = (uint32_t)a.n, total = (uint32_t)(a.n * a.k), T = (uint32_t)a.tokens;
  const int B = (int)a.batch, blocks = (int)(a.k * a.batch), e = blockIdx.x;
  int32_t* const R = route_mem;
  int32_t* const D = R + blocks + 1;
  int32_t* const C = D + blocks;
  const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));  // lanes below this one
  if (tid == 0) lower = valid = 0;  // behind the first step's barrier

  // One step: entries base + 512 * wave + 64 j + lane, j < 8.  mine(p, hit, r, v)
  // is called for each with its expert index v, whether that is e and its rank.
  // One barrier a step: the counts alternate between two buffers.
  int32_t carry = 0;
  int buf = 0;
  auto walk = [&](auto&& mine) __attribute__((always_inline)) {
    carry = 0;
    for (uint32_t base = 0; base < total; base += kRouteThreads * kRouteRun, buf ^= 1) {
      const uint32_t p0 = base + (uint32_t)(wave * 64 * kRouteRun + lane);
      int64_t v[kRouteRun];
#pragma unroll
      for (int j = 0; j < kRouteRun; ++j) {
        const uint32_t p = p0 + 64 * j, slot = p / n, tok = p - slot * n;
        v[j] = p < total ? a.index[(int64_t)tok * a.k + slot] : -1;
      }
      uint64_t hit[kRouteRun];
      int32_t hits = 0;
#pragma unroll
      for (int j = 0; j < kRouteRun; ++j) {
        hit[j] = __ballot(v[j] == e);
        hits += __popcll(hit[j]);
      }
      if (lane == 0) count[buf][wave] = hits;
      __syncthreads();
      int32_t r = carry;
#pragma unroll
      for (int w = 0; w < kRouteWaves; ++w) {
        const int32_t c = count[buf][w];
        if (w < wave) r += c;
        carry += c;
      }
#pragma unroll
      for (int j = 0; j < kRouteRun; ++j) {
        mine(p0 + 64 * j, v[j] == e, r + (int32_t)__popcll(hit[j] & lt), v[j]);
        r += (int32_t)__popcll(hit[j]);
      }
    }
  };

  int32_t low = 0, in = 0;
  walk([&](uint32_t p, bool, int32_t r, int64_t v) __attribute__((always_inline)) {
    low += v >= 0 && v < e;
    in += v >= 0 && v < a.experts;
    const uint32_t f = p / T;
    if (p < total && p == f * T) R[f] = r;
  });
  for (int off = 32; off; off >>= 1) {
    low += __shfl_xor(low, off, 64);
    in += __shfl_xor(in, off, 64);
  }
  if (lane == 0) {
    atomicAdd(&lower, low);
    atomicAdd(&valid, in);
  }
  if (tid == 0) R[blocks] = carry;
  __syncthreads();
  const int32_t off = lower;
  for (int b = tid; b < B; b += kRouteThreads) {
    int32_t c = 0;
    for (int f = b; f < blocks; f += B) c += R[f + 1] - R[f];
    C[b] = c;
  }
  __syncthreads();
  route_scan(C, B, wsum);
  int32_t* const seg = a.seg + (int64_t)e * (B + 1);
  for (int b = tid; b < B; b += kRouteThreads) {
    int32_t run = C[b];
    seg[b] = run;
    for (int f = b; f < blocks; f += B) {
      D[f] = run - R[f];
      run += R[f + 1] - R[f];
    }
  }
  if (tid == 0) {
    seg[B] = R[blocks];
    a.offsets[e] = off;
    if (e + 1 == (int)a.experts) a.offsets[a.experts] = valid;
  }
  __syncthreads();
  walk([&](uint32_t p, bool hit, int32_t r, int64_t) __attribute__((always_inline)) {
    if (!hit) return;
    a.entries[off + r] = (int32_t)p;
    a.rows[off + D[p / T] + r] = r;  // expert-local routed row
  });
}

// Ranks of this wave's 64 keys among equal keys of the wave (stable), one
// ballot per distinct key; r = lanes below with the same key, t = all of them.
__device__ __forceinline__ void route_ranks(bool ok, int key, uint64_t lt, int& r, int& t) {
  r = 0;
  t = 0;
  for (uint64_t act = __ballot(ok); act;) {
    const int ke = __builtin_amdgcn_readlane(key, __builtin_ctzll(act));
    const bool mine = ok && key == ke;
    const uint64_t m = __ballot(mine);
    if (mine) {
      r = __popcll(m & lt);
      t = __popcll(m);
    }
    act &= ~m;
  }
}

// seg and rows behind a by-expert sort (offsets, entries), for index matrices
// with more (slot, sample) blocks than moe_route_kernel holds: wave w of the
// grid takes expert e = w, counts its entries by sample, and walks them again
// (routed order) 64 at a time.  The per-sample counters sit in LDS (B ints per
// wave; up to 4 waves per workgroup, as many as keep them within 64 KB).
constexpr int kRowsWaves = 4;
__global__ __launch_bounds__(kRowsWaves * 64) void moe_route_rows(RouteArgs a) {
  extern __shared__ int32_t cnt_all[];  // (blockDim / 64) * B
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int e = blockIdx.x * (int)(blockDim.x >> 6) + wave;
  const int B = (int)a.batch;
  if (e >= a.experts) return;  // uniform per wave; no barrier below
  int32_t* cnt = cnt_all + wave * B;
  int32_t* const seg = a.seg + (int64_t)e * (B + 1);
  const int32_t o = a.offsets[e], oend = a.offsets[e + 1];
  const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));  // lanes below this one
  const uint32_t n = (uint32_t)a.n, T = (uint32_t)a.tokens;
  auto sample = [&](int32_t i) __attribute__((always_inline)) {  // token p % N, its sample
    const uint32_t p = (uint32_t)a.entries[i];
    return (int)((p - (p / n) * n) / T);
  };
  for (int b = lane; b < B; b += 64) cnt[b] = 0;
  __builtin_amdgcn_wave_barrier();
  for (int32_t i = o + lane; i < oend; i += 64) atomicAdd(&cnt[sample(i)], 1);
  __builtin_amdgcn_wave_barrier();
  int32_t run = 0;
  for (int b0 = 0; b0 < B; b0 += 64) {
    const int b = b0 + lane;
    const int32_t c = b < B ? cnt[b] : 0;
    int32_t x = c;  // inclusive over the wave
    for (int off = 1; off < 64; off <<= 1) {
      const int32_t y = __shfl_up(x, off, 64);
      if (lane >= off) x += y;
    }
    if (b < B) {
      seg[b] = run + x - c;
      cnt[b] = o + run + x - c;
    }
    run += __shfl(x, 63, 64);
  }
  if (lane == 0) seg[B] = run;
  __builtin_amdgcn_wave_barrier();
  for (int32_t base = o; base < oend; base += 64) {
    const int32_t i = base + lane;
    const bool ok = i < oend;
    const int b = ok ? sample(i) : 0;
    int r, t;
    route_ranks(ok, b, lt, r, t);
    const int32_t s2 = ok ? cnt[b] + r : 0;
    // every lane has read the counters before the last lane of each sample bumps them
    __builtin_amdgcn_wave_barrier();
    if (ok) {
      a.rows[s2] = i - o;  // expert-local routed row
      if (r == t - 1) cnt[b] = s2 + 1;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

}  // namespace
}  // namespace da

extern "C" {

int da_moe_topk(const void* logits, int dtype, int64_t n_tokens, int n_experts, int k,
                int64_t row_stride, float* weights, int64_t* index, void* stream) {
  using namespace da;
  const char* who = "da_moe_topk";
  if (!valid_dtype(dtype)) return set_error(DA_ERR_INVALID, "%s: bad dtype", who);
  if (n_tokens < 0) return set_error(DA_ERR_INVALID, "%s: negative token count", who);
  if (n_experts < 1 || n_experts > kMaxExperts)
    return set_error(DA_ERR_INVALID, "%s: n_experts must be in [1, %d]", who, kMaxExperts);
  if (k < 1 || k > n_experts || k > kMaxTopK)
    return set_error(DA_ERR_INVALID, "%s: k must be in [1, min(n_experts, %d)]", who, kMaxTopK);
  if (row_stride < n_experts) return set_error(DA_ERR_INVALID, "%s: row stride < n_experts", who);
  if (n_tokens == 0) return DA_OK;
  if (!logits || !weights || !index) return set_error(DA_ERR_INVALID, "%s: NULL pointer", who);
  const int lanes = n_experts <= 128 ? kWave : kWave / 2;
  if ((n_tokens + lanes - 1) / lanes > 0x7fffffffLL) return set_error(DA_ERR_INVALID, "%s: too many tokens", who);
  const unsigned blocks = (unsigned)((n_tokens + lanes - 1) / lanes);
  const size_t lds = (size_t)n_experts * lanes * (sizeof(float) + sizeof(uint16_t)) + (size_t)k * lanes * sizeof(float);
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case DA_BF16: moe_topk_kernel<DA_BF16><<<blocks, lanes, lds, st>>>((const char*)logits, n_tokens, n_experts, k, row_stride, weights, index); break;
    case DA_F16: moe_topk_kernel<DA_F16><<<blocks, lanes, lds, st>>>((const char*)logits, n_tokens, n_experts, k, row_stride, weights, index); break;
    default: moe_topk_kernel<DA_F32><<<blocks, lanes, lds, st>>>((const char*)logits, n_tokens, n_experts, k, row_stride, weights, index); break;
  }
  return check_launch(who);
}

int da_counting_sort(const int32_t* keys32, const int64_t* keys64, int64_t n, int64_t rows,
                     int64_t k, int slot_major, int64_t key_div, int bins, int32_t* offsets,
                     int32_t* perm, void* stream) {
  using namespace da;
  const char* who = "da_counting_sort";
  if (n < 0 || bins < 1 || bins > kMaxBins)
    return set_error(DA_ERR_INVALID, "%s: need n >= 0 and 1 <= bins <= %d", who, kMaxBins);
  if (n > 0x7fffffffLL) return set_error(DA_ERR_INVALID, "%s: at most 2^31-1 entries", who);
  if (key_div < 1) return set_error(DA_ERR_INVALID, "%s: key_div must be >= 1", who);
  if (slot_major) {
    if (!keys64 || rows < 1 || k < 1 || rows * k != n)
      return set_error(DA_ERR_INVALID, "%s: slot-major keys need an int64 (rows, k) matrix with rows*k == n", who);
  } else if (n > 0 && !keys32 && !keys64) {
    return set_error(DA_ERR_INVALID, "%s: no keys", who);
  }
  if (!offsets || (n > 0 && !perm)) return set_error(DA_ERR_INVALID, "%s: NULL output", who);
  SortArgs a;
  a.keys32 = keys32;
  a.keys64 = keys64;
  a.n = n;
  a.rows = rows;
  a.k = k;
  a.slot_major = slot_major;
  a.bins = bins;
  a.offsets = offsets;
  a.perm = perm;
  a.key_div = key_div;
  counting_sort_kernel<<<1, 256, 0, (hipStream_t)stream>>>(a);
  return check_launch(who);
}

int da_moe_route(const int64_t* index, int64_t n_tokens, int k, int n_experts, int64_t batch,
                 int64_t tokens, int32_t* expert_offsets, int32_t* entries, int32_t* seg, int32_t* rows,
                 void* stream) {
  using namespace da;
  const char* who = "da_moe_route";
  if (n_tokens < 0 || k < 1 || k > kMaxTopK)
    return set_error(DA_ERR_INVALID, "%s: need n_tokens >= 0 and 1 <= k <= %d", who, kMaxTopK);
  if (n_experts < 1 || n_experts > kMaxExperts)
    return set_error(DA_ERR_INVALID, "%s: n_experts must be in [1, %d]", who, kMaxExperts);
  if (batch < 1 || tokens < 1 || batch * tokens != n_tokens)
    return set_error(DA_ERR_INVALID, "%s: n_tokens must equal batch * tokens", who);
  if ((int64_t)n_experts * batch > kMaxBins)
    return set_error(DA_ERR_INVALID, "%s: n_experts * batch must be <= %d", who, kMaxBins);
  if (n_tokens * k > 0x7fffffffLL) return set_error(DA_ERR_INVALID, "%s: at most 2^31-1 entries", who);
  if (!index || !expert_offsets || !entries || !seg || !rows)
    return set_error(DA_ERR_INVALID, "%s: NULL pointer", who);
  RouteArgs a;
  a.index = index;
  a.n = n_tokens;
  a.k = k;
  a.experts = n_experts;
  a.batch = batch;
  a.tokens = tokens;
  a.offsets = expert_offsets;
  a.entries = entries;
  a.seg = seg;
  a.rows = rows;
  hipStream_t st = (hipStream_t)stream;
  if ((int64_t)k * batch <= kRouteBlocks) {
    const size_t lds = route_lds((int64_t)k * batch, batch);  // <= 96 KB
    if (lds > 48 * 1024) {
      // Idempotent, so racing first calls are harmless.
      static std::atomic<bool> attr_set{false};
      if (!attr_set.load(std::memory_order_relaxed)) {
        if (hipFuncSetAttribute((const void*)moe_route_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)route_lds(kRouteBlocks, kMaxBins)) != hipSuccess)
          return set_error(DA_ERR_HIP, "%s: hipFuncSetAttribute failed", who);
        attr_set.store(true, std::memory_order_relaxed);
      }
    }
    moe_route_kernel<<<(unsigned)n_experts, kRouteThreads, lds, st>>>(a);
    return check_launch(who);
  }
  const int rc = da_counting_sort(nullptr, index, n_tokens * k, n_tokens, k, 1, 1, n_experts, expert_offsets, entries,
                                  stream);
  if (rc) return rc;
  const int waves = batch <= 4096 ? kRowsWaves : 2;  // batch <= 8192: at most 64 KB of counters
  const unsigned blocks = (unsigned)((n_experts + waves - 1) / waves);
  moe_route_rows<<<blocks, waves * 64, (size_t)waves * batch * sizeof(int32_t), st>>>(a);
  return check_launch(who);
}

int da_compact_rows(const uint8_t* mask, int64_t batch, int64_t tokens, int32_t* seg_offsets, int32_t* rows,
                    void* stream) {
  using namespace da;
  const char* who = "da_compact_rows";
  if (batch < 0 || tokens < 0) return set_error(DA_ERR_INVALID, "%s: negative size", who);
  if (batch * tokens > 0x7fffffffLL) return set_error(DA_ERR_INVALID, "%s: at most 2^31-1 rows", who);
  if (!seg_offsets || (batch * tokens > 0 && (!mask || !rows)))
    return set_error(DA_ERR_INVALID, "%s: NULL pointer", who);
  compact_rows_kernel<<<1, 1024, 0, (hipStream_t)stream>>>(mask, batch, tokens, seg_offsets, rows);
  return check_launch(who);
}

}  // extern "C"
