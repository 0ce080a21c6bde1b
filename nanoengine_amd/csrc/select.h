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

// 4096 bins for the scores of keys kmin to kmax: positive ones linear in the key
// (an outlier or a long tail then costs a few octaves of bins), ones that cross
// zero linear in the score. One type, chosen at run time: with an instantiation
// of the list select for each, its usual path took 15.3 us for 14.2.
struct ListBins {
  ScoreBins scores;
  KeyBins keys;
  bool linear;
  __device__ __forceinline__ ListBins(uint32_t kmin, uint32_t kmax, uint32_t score_max)
      : scores(kmin, score_max), keys(kmin, kmax), linear(kmin <= order_key(0.f)) {}
  __device__ __forceinline__ ListBins(uint32_t kmin, uint32_t kmax) : ListBins(kmin, kmax, kmax) {}
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

// Adds one to hist[d] for every calling lane; where half of a wave shares the
// first lane's bin (ties), one atomic for those: on one LDS word they would go
// one after another.
__device__ __forceinline__ void crowd_add(uint32_t* hist, uint32_t d) {
  const uint32_t first = __builtin_amdgcn_readfirstlane(d);  // of the lanes here
  const uint64_t same = __ballot(d == first);
  const uint32_t n = (uint32_t)__popcll(same);
  const bool share = n >= 32 && d == first;
  if (!share || (int)(threadIdx.x & 63) == __builtin_ctzll(same)) atomicAdd(&hist[d], share ? n : 1u);
}

// The smallest and largest of the block's values (NT threads), to all of them;
// returns the lowest of the waves' largest.
template <int NT>
__device__ __forceinline__ uint32_t block_range(uint32_t* wave_sum, uint32_t& low, uint32_t& high) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    low = min(low, (uint32_t)__shfl_xor(low, off, 64));
    high = max(high, (uint32_t)__shfl_xor(high, off, 64));
  }
  if (lane == 0) {
    wave_sum[wave] = low;
    wave_sum[NT / 64 + wave] = high;
  }
  __syncthreads();
  uint32_t least = 0xffffffffu;
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) {
    low = min(low, wave_sum[i]);
    high = max(high, wave_sum[NT / 64 + i]);
    least = min(least, wave_sum[NT / 64 + i]);
  }
  return least;
}

// Of the elements with keys in [kmin, kmax], too many to rank by counting, the
// `remain` first ones (fewer than there are) are marked: the range is binned
// again (outliers and long tails leave most scores in one bin), the threshold
// bin ranked if that leaves it few elements, and otherwise (ties) radix levels
// follow over what it spans. pass(f) calls f(key, position) for every element of
// the row, in or out of the range; mark(position) selects one; ties(key, n) may
// mark the n lowest positions of one key by itself (true), else the levels do.
// Bins: the second binning (two kinds of bins at run time cost rows of 8K with an
// outlier 1 us).
// s holds the block's hist, wave_sum, rank, tb, above, eq and a count that is 0
// on entry. All threads call it, with the same arguments.
template <int NT, typename Bins, typename Smem, typename Pass, typename Mark, typename Ties>
__device__ __forceinline__ void select_crowd(Smem& s, uint32_t kmin, uint32_t kmax, uint32_t remain, Pass&& pass,
                                             Mark&& mark, Ties&& ties) {
  const int tid = threadIdx.x, lane = tid & 63;
  auto each = [&](auto&& f) {
    pass([&](uint32_t key, uint32_t pos) {
      if (key >= kmin && key <= kmax) f(key, pos);
    });
  };
  if (kmin != kmax) {
    for (int i = tid; i < kHistBins; i += NT) s.hist[i] = 0u;
    // -inf, alone below every other score, must not stretch the range
    const uint32_t ninf = order_key(-__builtin_inff());
    uint32_t low = kmin, high = kmax;
    if (kmin <= ninf) {
      low = 0xffffffffu;
      each([&](uint32_t key, uint32_t) { low = min(low, key > ninf ? key : 0xffffffffu); });
      __syncthreads();  // every thread has read the range
      block_range<NT>(s.wave_sum, low, high);
    }
    __syncthreads();
    const Bins bins(low, min(high, order_key(3.4028235e38f)));
    uint32_t lowest = 0;
    each([&](uint32_t key, uint32_t) {
      const uint32_t d = bins.of(key);
      if (d) crowd_add(s.hist, d);
      else ++lowest;
    });
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) lowest += (uint32_t)__shfl_xor(lowest, off, 64);
    if (lane == 0 && lowest) atomicAdd(&s.hist[0], lowest);
    __syncthreads();
    find_threshold<NT>(s.hist, s.wave_sum, kHistBins, remain, &s.tb, &s.above, &s.eq);
    const uint32_t tb = s.tb, eq = s.eq;
    remain -= s.above;
    const bool whole_bin = eq == remain, ranked = !whole_bin && eq <= (uint32_t)kRankCap;
    low = 0xffffffffu;
    high = 0u;
    each([&](uint32_t key, uint32_t pos) {
      const uint32_t d = bins.of(key);
      if (d > tb || (whole_bin && d == tb)) {
        mark(pos);
      } else if (d == tb) {
        if (ranked) {
          s.rank[atomicAdd(&s.count, 1u)] = rank_composite(key, pos);
        } else {
          low = min(low, key);
          high = max(high, key);
        }
      }
    });
    __syncthreads();
    if (whole_bin) return;
    if (ranked) {
      if ((uint32_t)tid < eq) {
        const uint64_t mine = s.rank[tid];
        uint32_t ahead = 0;
        for (uint32_t j = 0; j < eq; ++j) ahead += s.rank[j] > mine ? 1u : 0u;
        if (ahead < remain) mark(kIdxMax - (uint32_t)(mine & kIdxMax));
      }
      return;
    }
    block_range<NT>(s.wave_sum, low, high);
    kmin = low;
    kmax = high;
  }
  if (kmin == kmax && ties(kmin, remain)) return;
  const CompositeDigits digits(kmin, kmax);
  uint64_t prefix = 0;  // the digits chosen so far
  for (int L = 0; L < digits.levels; ++L) {
    __syncthreads();  // every thread has read the previous level's outcome
    for (int i = tid; i < digits.bins(L); i += NT) s.hist[i] = 0u;
    __syncthreads();
    each([&](uint32_t key, uint32_t pos) {
      if (digits.above(key, pos, L) == prefix) crowd_add(s.hist, digits.of(key, pos, L));
    });
    __syncthreads();
    find_threshold<NT>(s.hist, s.wave_sum, digits.bins(L), remain, &s.tb, &s.above, &s.eq);
    const uint32_t t = s.tb;
    remain -= s.above;
    const bool done = s.eq == remain || L == digits.levels - 1;
    each([&](uint32_t key, uint32_t pos) {
      const uint32_t d = digits.of(key, pos, L);
      if (digits.above(key, pos, L) == prefix && (d > t || (done && d == t))) mark(pos);
    });
    if (done) return;
    prefix = prefix * (uint32_t)digits.bins(L) + t;
  }
}

}  // namespace dsa
