// Device helpers of the exact selects: key and score conversion, the linear
// score bins, the block scan and the composite rank (gfx950).
#pragma once

#include "dsa_common.h"

namespace dsa {

constexpr int kHistBins = 4096;
constexpr uint32_t kIdxMax = (1u << 18) - 1;  // positions are at most this
constexpr int kRankCap = 384;                 // threshold-bin candidates ranked by counting

// (score, lower position first) as one integer: every element is distinct.
__device__ __forceinline__ uint64_t rank_composite(uint32_t key, uint32_t pos) {
  return ((uint64_t)key << 18) | (kIdxMax - pos);
}

// Inverse of order_key: the float whose key is k.
__device__ __forceinline__ float key_to_float(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k ^ 0x80000000u) : ~k);
}

// Exclusive block prefix sum of one value per thread; returns the prefix and
// writes the block total to *total (all threads).
template <int NT>
__device__ uint32_t block_exclusive_scan(uint32_t* wave_sum, uint32_t x, uint32_t* total) {
  constexpr int kWaves = NT / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t v = x;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    uint32_t n = __shfl_up(v, off, 64);
    if (lane >= off) v += n;
  }
  __syncthreads();
  if (lane == 63) wave_sum[wave] = v;
  __syncthreads();
  uint32_t before = 0, all = 0;
  for (int w = 0; w < kWaves; ++w) {
    uint32_t t = wave_sum[w];
    if (w < wave) before += t;
    all += t;
  }
  *total = all;
  return before + v - x;
}

// 4096 bins linear in the score between the scores of keys kmin and kmax. The
// bin never decreases with the key (subtraction, multiplication by a positive
// scale and truncation are each monotone, +-0 share a bin), so a candidate in
// a higher bin ranks ahead. Scores that are not finite, or whose range is not,
// fall into the end bins or all into one.
struct ScoreBins {
  float lo, scale;
  __device__ __forceinline__ ScoreBins(float lowest, float highest) {
    lo = lowest;
    const float range = highest - lowest;
    scale = range > 0.f && range < __builtin_inff() ? (float)(kHistBins - 1) / range : 0.f;
  }
  __device__ __forceinline__ ScoreBins(uint32_t kmin, uint32_t kmax)
      : ScoreBins(key_to_float(kmin), key_to_float(kmax)) {}
  __device__ __forceinline__ uint32_t bin(float score) const {
    const float x = (score - lo) * scale;  // NaN (inf * 0) maps to bin 0
    return (uint32_t)fminf(fmaxf(x, 0.f), (float)(kHistBins - 1));
  }
  __device__ __forceinline__ uint32_t of(uint32_t key) const { return bin(key_to_float(key)); }
};

// 4096 bins linear in the bits of the scores from `lowest` > 0 to `highest`
// (positive floats order as their bits); lower scores share bin 0, higher ones
// the last.
struct BitBins {
  float lo;
  uint32_t base;
  int shift;
  __device__ __forceinline__ BitBins(float lowest, float highest) {
    const float top = fmaxf(highest, lowest);
    lo = lowest;
    base = __float_as_uint(lowest);
    shift = max(0, 32 - (int)__clz((int)(__float_as_uint(top) - base)) - 12);
  }
  __device__ __forceinline__ uint32_t bin(float score) const {
    return score < lo ? 0u : min((__float_as_uint(score) - base) >> shift, (uint32_t)(kHistBins - 1));
  }
};

// The same on order keys: 4096 bins linear in the key from kmin to kmax; lower
// keys share bin 0, higher ones the last.
struct KeyBins {
  uint32_t base;
  int shift;
  __device__ __forceinline__ KeyBins(uint32_t kmin, uint32_t kmax)
      : base(kmin), shift(max(0, 32 - (int)__clz((int)(max(kmin, kmax) - kmin)) - 12)) {}
  __device__ __forceinline__ uint32_t of(uint32_t key) const {
    return key < base ? 0u : min((key - base) >> shift, (uint32_t)(kHistBins - 1));
  }
};

// 4096 bins for the scores of keys kmin to kmax: positive ones linear in the
// key; ones that cross zero linear in the score, unless the largest is far above
// the lowest's magnitude (an outlier, a long tail), where the 40 octaves below
// it take the bins. One type, chosen at run time: an instantiation of the list
// select for each would run its code cold.
struct ListBins {
  ScoreBins scores;
  KeyBins keys;
  bool linear;
  __device__ __forceinline__ ListBins(uint32_t kmin, uint32_t kmax)
      : scores(kmin, kmax), keys(kmin, kmax), linear(false) {
    if (kmin > order_key(0.f)) return;
    const float lo = key_to_float(kmin), hi = key_to_float(kmax);
    if (hi > -16.f * lo) keys = KeyBins(order_key(hi * 0x1p-40f), kmax);
    else linear = true;
  }
  __device__ __forceinline__ uint32_t of(uint32_t key) const {
    const uint32_t a = scores.of(key), b = keys.of(key);
    return linear ? a : b;
  }
};

// The 12-bit digits, from the top, of the composites of keys in [kmin, kmax]:
// the key part counts from kmin, so the digits spread over the keys' own range.
struct CompositeDigits {
  uint32_t kmin;
  int total_bits, levels;
  __device__ __forceinline__ CompositeDigits(uint32_t lo, uint32_t hi)
      : kmin(lo), total_bits(32 - __clz(hi - lo) + 18), levels((total_bits + 11) / 12) {}
  __device__ __forceinline__ int bins(int level) const {
    const int top = total_bits - 12 * level;
    return 1 << (top - max(top - 12, 0));
  }
  // the digits above `level`, as one number
  __device__ __forceinline__ uint64_t above(uint32_t key, uint32_t pos, int level) const {
    return rank_composite(key - kmin, pos) >> (total_bits - 12 * level);
  }
  __device__ __forceinline__ uint32_t of(uint32_t key, uint32_t pos, int level) const {
    const int top = total_bits - 12 * level;
    const int lo_b = max(top - 12, 0);
    return (uint32_t)((rank_composite(key - kmin, pos) >> lo_b) & ((1ull << (top - lo_b)) - 1ull));
  }
};

}  // namespace dsa
