// fp32 operands on the 16-bit matrix pipe.
//
// An fp32 value is exactly the sum of three bf16 values: hi = bf16(x), mid =
// bf16(x - hi), lo = x - hi - mid (8 + 8 + 8 significant bits, each rounded to
// nearest, so mid and lo may be negative).  A product of two fp32 values is then
// hi*hi + (hi*mid + mid*hi) + (hi*lo + mid*mid + lo*hi) up to terms below 2^-24
// of it, every one of them exact in the fp32 accumulator's multiplier: six bf16
// products per fp32 one.  v_mfma_f32_32x32x16_bf16 does 16 times the work of
// v_mfma_f32_32x32x2_f32 per pass, so the six still leave 2.7 times the rate,
// and the sums are rounded fewer times (per 16 terms instead of 2), the small
// products first.
//
// A pre-pass writes rows [hi | mid | lo], each part padded with zeros to whole
// 128-byte stages (6 bytes written per 4 read, HBM-bound); the tile kernels
// then run their 2-byte engine over six (part, part) segments.  Infinities, NaN,
// magnitudes below 2^-100 but not zero (lo could be subnormal) and those from
// 2^50 raise a flag: the split kernels then return at once and the fp32 kernels,
// launched behind them and otherwise returning at once, do the whole call.
// Under 2^50 no sum of up to 2^27 products leaves the fp32 range.  Where one
// does, the parts overflow on their own and in their own order: hi*mid, with mid
// of either sign, is infinite from 2^8 past the range, and -inf + inf is NaN
// where an fp32 product is +inf.
#pragma once

#include "common.h"

namespace da {
namespace {
namespace split {

constexpr int kMaxMats = 40;  // matrices per launch
constexpr int kSegs = 6;
// (side 1 part, side 2 part) of the segments, two bits each, small products first.
constexpr uint32_t kPart1 = 2u | 0u << 2 | 1u << 4 | 1u << 6 | 0u << 8 | 0u << 10;
constexpr uint32_t kPart2 = 0u | 2u << 2 | 1u << 4 | 0u << 6 | 1u << 8 | 0u << 10;

// Elements of one part of a row of `width` fp32 values: whole 128-byte stages.
inline int64_t part_elems(int64_t width) { return (width + 63) / 64 * 64; }
inline int64_t row_bytes(int64_t width) { return 3 * part_elems(width) * 2; }

struct Mat {
  const char* src;
  char* dst;
  const int32_t* index;       // row r is source row index[r] (null: r)
  const int32_t* live;        // rows past *live are left out (null: none)
  int64_t rows, tokens;       // source row s: sample s / tokens, token s % tokens (indexed rows: all of sample 0)
  int64_t bstride, tstride;   // bytes
  int64_t width;              // the source's width, elements (a multiple of 4)
  int32_t chunks, chunks_in;  // 8-element chunks per part and those the source fills
  int64_t block0;
};
struct Args {
  Mat mats[kMaxMats];
  int n;
  uint32_t* flag;
};
static_assert(sizeof(Args) <= 4096, "kernel arguments");

// A tile kernel with a gate runs only when (*flag != 0) == on.
struct Gate {
  const uint32_t* flag;
  uint32_t on;
};
__device__ __forceinline__ bool gate_closed(const Gate& g) { return g.flag && (*g.flag != 0u) != (g.on != 0u); }

// The segment of stage s of a loop with nk stages per part, and the byte
// offsets of that stage in rows of either side.
struct Offsets {
  uint32_t k1, k2;
};
__device__ __forceinline__ int segment(int s, int nk) {
  return (s >= nk) + (s >= 2 * nk) + (s >= 3 * nk) + (s >= 4 * nk) + (s >= 5 * nk);
}
__device__ __forceinline__ Offsets offsets(int s, int nk, uint32_t part_bytes) {
  const int seg = segment(s, nk);
  const uint32_t k = (uint32_t)(s - seg * nk) * 128u;
  return Offsets{k + ((kPart1 >> (2 * seg)) & 3u) * part_bytes, k + ((kPart2 >> (2 * seg)) & 3u) * part_bytes};
}

__device__ __forceinline__ bool outside(float x) {
  const uint32_t e = (__float_as_uint(x) >> 23) & 0xffu;
  return (e >= 127u + 50u) | ((e < 127u - 100u) & (x != 0.f));
}

// One thread: 8 values of one row.  Values in range round to finite parts; the
// ones that raise the flag are written as they come out and never read.
__global__ __launch_bounds__(256) void split_rows(Args a) {
  int i = 0;
  while (i + 1 < a.n && a.mats[i + 1].block0 <= (int64_t)blockIdx.x) ++i;
  const Mat& m = a.mats[i];
  const int64_t idx = ((int64_t)blockIdx.x - m.block0) * 256 + threadIdx.x;
  const int64_t r = idx / m.chunks;
  const int c = (int)(idx - r * m.chunks);
  if (r >= m.rows || (m.live && r >= *m.live)) return;
  const int64_t sr = m.index ? m.index[r] : r;
  uint32_t part[3][4] = {};
  bool bad = false;
  if (c < m.chunks_in) {
    const char* p = m.src + (sr / m.tokens) * m.bstride + (sr % m.tokens) * m.tstride + (int64_t)c * 32;
    float x[8];
    const u32x4 v0 = __builtin_nontemporal_load((const u32x4*)p);
    // a width of 4 mod 8 ends with half a chunk
    const u32x4 v1 = 8 * c + 4 < m.width ? __builtin_nontemporal_load((const u32x4*)p + 1) : u32x4{0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[e] = __uint_as_float(v0[e]);
      x[4 + e] = __uint_as_float(v1[e]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      bad |= outside(x[e]);
      const uint32_t hi = f32_to_bf16_bits(x[e]);
      const float r1 = x[e] - bf16_bits_to_f32(hi);
      const uint32_t mid = f32_to_bf16_bits(r1);
      const uint32_t lo = f32_to_bf16_bits(r1 - bf16_bits_to_f32(mid));
      const int sh = 16 * (e & 1);
      part[0][e >> 1] |= hi << sh;
      part[1][e >> 1] |= mid << sh;
      part[2][e >> 1] |= lo << sh;
    }
  }
  char* d = m.dst + (r * 3 * m.chunks + c) * 16;
#pragma unroll
  for (int q = 0; q < 3; ++q)
    st16(d + (int64_t)q * m.chunks * 16, u32x4{part[q][0], part[q][1], part[q][2], part[q][3]});
  if (bad) atomicOr(a.flag, 1u);
}

// A call's time in us on fp32 rows and on split ones.  Its workgroups run
// `fp32_stages` and `stages` 128-byte stages of a 256 x 128 tile in all, the
// longest chain of one workgroup longest32 / longest; a stage takes about 4.0 us
// on the fp32 matrix pipe (1102 tiles of 120 stages: 2396 us) and 0.95 us on the
// bf16 one.  The pre-pass moves 10 bytes per value at about 5 TB/s.
struct Cost {
  double stages32 = 0, stages = 0, longest32 = 0, longest = 0, values = 0;
  void tiles(double n, int64_t width, double fp32_us) {
    const double s32 = (double)((width + 31) / 32) * fp32_us, s = (double)(kSegs * part_elems(width) / 64) * 0.95;
    chain32_ += s32;
    chain_ += s;
    stages32 += n * s32;
    stages += n * s;
  }
  void end_chain() {
    longest32 = chain32_ > longest32 ? chain32_ : longest32;
    longest = chain_ > longest ? chain_ : longest;
    chain32_ = chain_ = 0;
  }
  bool pays(int64_t slots) const {
    const double a = stages32 / (double)slots, b = stages / (double)slots;
    return (b > longest ? b : longest) + values * 10.0 / 5e6 + 10.0 < 0.95 * (a > longest32 ? a : longest32);
  }

 private:
  double chain32_ = 0, chain_ = 0;
};
constexpr size_t kMaxBytes = (size_t)4 << 30;  // the split copies of one call

// Collects the matrices of a call, lays their split copies out behind `ws` and
// launches the pre-pass.  A matrix given twice (one block on both sides) is
// split once.
class Builder {
 public:
  Builder(char* ws, hipStream_t st) : flag_((uint32_t*)ws), next_(ws ? ws + 256 : nullptr), st_(st) { args_.n = 0; }

  // Bytes one matrix takes.
  static size_t bytes(int64_t rows, int64_t width) { return ((size_t)(rows * row_bytes(width)) + 255) / 256 * 256; }

  // Where the split rows of `rows` = batch * tokens rows go: row r at r * row_bytes(width).
  char* add(const void* src, int64_t batch, int64_t tokens, int64_t bstride, int64_t tstride, int64_t width,
            const int32_t* index = nullptr, const int32_t* live = nullptr) {
    // An index names rows of the capture behind the side, also past the `tokens` packed ones.
    const int64_t per_sample = index ? INT64_MAX : tokens > 0 ? tokens : 1;
    for (int i = 0; i < n_; ++i) {
      const Mat& m = seen_[i];
      if (m.src == src && m.index == index && m.live == live && m.rows == batch * tokens && m.tokens == per_sample &&
          m.bstride == bstride && m.tstride == tstride && m.width == width)
        return m.dst;
    }
    if (args_.n == kMaxMats) flush();
    Mat m;
    m.src = (const char*)src;
    m.dst = next_;
    m.index = index;
    m.live = live;
    m.rows = batch * tokens;
    m.tokens = per_sample;
    m.bstride = bstride;
    m.tstride = tstride;
    m.chunks = (int32_t)(part_elems(width) / 8);
    m.chunks_in = (int32_t)((width + 7) / 8);
    m.width = width;
    m.block0 = blocks_;
    next_ += bytes(m.rows, width);
    blocks_ += (m.rows * m.chunks + 255) / 256;
    args_.mats[args_.n++] = m;
    if (n_ < kMaxMats) seen_[n_++] = m;
    return m.dst;
  }
  // Clears the flag (first) and splits what has been added.
  int flush() {
    if (rc_ == 0 && !cleared_) {
      rc_ = zero_f32_2d((float*)flag_, 1, 1, 1, st_);
      cleared_ = true;
    }
    args_.flag = flag_;
    if (rc_ == 0 && blocks_ > 0) {
      split_rows<<<(unsigned)blocks_, 256, 0, st_>>>(args_);
      rc_ = check_launch("split_rows");
    }
    args_.n = 0;
    blocks_ = 0;
    return rc_;
  }
  const uint32_t* flag() const { return flag_; }

 private:
  uint32_t* flag_;
  char* next_;
  hipStream_t st_;
  Args args_;
  Mat seen_[kMaxMats];
  int n_ = 0;
  int64_t blocks_ = 0;
  bool cleared_ = false;
  int rc_ = 0;
};

}  // namespace split
}  // namespace
}  // namespace da
