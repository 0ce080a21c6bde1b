// Exact top-k selection (+ page-table translation) and the logical->physical
// index transform for the DSA decode path, written for gfx950.
//
// Order: a most-significant-digit radix select on a 50-bit composite key
//   [ order_key(score) : 32 bits ][ (2^18-1) - position : 18 bits ]
// so that every element is distinct and equal scores resolve to the lowest
// positions (NaN ranks as -inf). Digits are 12/10/10 bits of the score key and
// 9/9 bits of the inverted position.
//
// Aligned rows of at most 64K positions take one launch (topk_row_kernel: the
// row in registers, binned by score). Longer, ragged or unaligned rows take
// three launches on the caller's stream:
//   1. threshold (one workgroup per row): a 1/8 sample of the row (contiguous
//      1024-element chunks, one in eight) gives, by a two-digit radix on the
//      sample, a score threshold t with about k + 4 sqrt(k) elements expected
//      at or above it - a bound that holds with a wide margin;
//   2. gather (8192 positions per workgroup, 8 per 64K row): one coalesced
//      read of the scores, one compare per element, and the elements at or
//      above t are appended - (key, position) - to the row's candidate list in
//      the workspace (wave ballots into LDS, one global atomic per workgroup);
//   3. finish (one workgroup per row): if the list holds between k and its
//      capacity entries, the exact top-k of the row is the exact top-k of the
//      list, found by radix levels in LDS; otherwise the row falls back to
//      the full exact select, which re-reads the row from HBM per level and
//      needs no bound at all. The selected positions are marked in an LDS
//      bitmap, compacted with one block prefix scan (ascending order, so the
//      output is deterministic) and written with the page translation.
// No global sort, no bounded candidate buffer on the exact path. The row
// select and the fused indexer's list select (topk_list_kernel) take a bin of
// the score as their first digit.
#include <mutex>

#include "dsa_common.h"
#include "indexer_page.h"
#include "select.h"
#include "../../include/dsa_amd.h"

namespace dsa {

constexpr int kTopkThreads = 512;
constexpr int kTopkMaxLen = 1 << 18;            // positions per row
constexpr int kBitmapWords = kTopkMaxLen / 32;  // 32 KB of LDS
constexpr int kLevels = 5;

// threshold / gather geometry
constexpr int kAuxThreads = 256;
constexpr int kSampleChunk = 1024;              // contiguous sampled chunk
constexpr int kSampleEvery = 8;                 // one chunk in eight
constexpr int kGatherPerThread = 32;
constexpr int kGatherSpan = kAuxThreads * kGatherPerThread;  // 8192 positions per workgroup
constexpr int kGatherLdsCap = 2048;             // candidates one gather workgroup can stage

struct TopkSmem {
  uint32_t hist[kHistBins];
  uint32_t bitmap[kBitmapWords];
  uint32_t list_key[2][kListCap];
  uint32_t list_pos[2][kListCap];
  uint32_t wave_sum[16];
  uint32_t list_count[2];
  uint32_t tb, above, eq;
};
constexpr size_t kTopkSmemBytes = sizeof(TopkSmem);

// LDS of the list select (two workgroups fit on a CU). A row the kernel repairs
// itself uses TopkSmem.
struct ListSmem {
  uint32_t hist[kHistBins];
  uint32_t bitmap[kBitmapWords];
  uint64_t rank[kRankCap];
  uint32_t wave_sum[16];
  uint32_t count, tb, above, eq;
};
static_assert(sizeof(ListSmem) <= sizeof(TopkSmem), "a repairing launch covers the list layout");

__device__ __forceinline__ uint32_t radix_digit(int level, uint32_t key, uint32_t pos) {
  switch (level) {
    case 0: return key >> 20;
    case 1: return (key >> 10) & 1023u;
    case 2: return key & 1023u;
    case 3: return ((kIdxMax - pos) >> 9) & 511u;
    default: return (kIdxMax - pos) & 511u;
  }
}

__device__ __forceinline__ int radix_bins(int level) {
  return level == 0 ? 4096 : (level < 3 ? 1024 : 512);
}

// Does (key, pos) carry the chosen digits of every level before `level`?
__device__ __forceinline__ bool in_bucket(int level, uint32_t key, uint32_t pos, const uint32_t* thr) {
  switch (level) {
    case 0: return true;
    case 1: return (key >> 20) == thr[0];
    case 2: return (key >> 10) == ((thr[0] << 10) | thr[1]);
    case 3: return key == ((thr[0] << 20) | (thr[1] << 10) | thr[2]);
    default:
      return key == ((thr[0] << 20) | (thr[1] << 10) | thr[2]) && (((kIdxMax - pos) >> 9) == thr[3]);
  }
}

// Positions of the set bits of bitmap[0, nwords) in ascending order into
// sel[0, top_k) (*total = all set bits). Thread t owns the 16-byte-aligned
// word range [4 q t, 4 q (t + 1)), q = ceil(nwords / 4NT), read with 16-byte
// loads (lanes 4q words apart: at most 2-way bank conflicts, where single
// words would conflict q-ways) and kept in registers for the second pass;
// words at or past nwords count as zero. Ends with a barrier.
template <int NT>
__device__ void compact_bitmap(const uint32_t* bitmap, int nwords, uint32_t* wave_sum, uint32_t* sel, int top_k,
                               uint32_t* total_out) {
  constexpr int kMaxQ = kBitmapWords / (4 * NT);
  static_assert(kMaxQ >= 1 && kBitmapWords % (4 * NT) == 0, "bitmap words per thread");
  const int tid = threadIdx.x;
  const int q = (nwords + 4 * NT - 1) / (4 * NT);
  const int w0 = tid * 4 * q;
  uint32_t v[4 * kMaxQ];
  uint32_t cnt = 0;
#pragma unroll
  for (int i = 0; i < kMaxQ; ++i) {
    uint4 x = {0u, 0u, 0u, 0u};
    if (i < q && w0 + 4 * i < nwords) x = *reinterpret_cast<const uint4*>(bitmap + w0 + 4 * i);
    v[4 * i] = x.x;
    v[4 * i + 1] = w0 + 4 * i + 1 < nwords ? x.y : 0u;
    v[4 * i + 2] = w0 + 4 * i + 2 < nwords ? x.z : 0u;
    v[4 * i + 3] = w0 + 4 * i + 3 < nwords ? x.w : 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k) cnt += __popc(v[4 * i + k]);
  }
  uint32_t total = 0;
  uint32_t at = block_exclusive_scan<NT>(wave_sum, cnt, &total);
  __syncthreads();  // sel may alias buffers read before this call
#pragma unroll
  for (int k = 0; k < 4 * kMaxQ; ++k) {
    uint32_t bits = v[k];
    while (bits) {
      const int bit = __ffs(bits) - 1;
      bits &= bits - 1;
      if (at < (uint32_t)top_k) sel[at] = (uint32_t)(((w0 + k) << 5) + bit);
      ++at;
    }
  }
  __syncthreads();
  *total_out = total;
}

// The same from byte flags (one per position, 0 or 1, flags[0, len) padded
// with zeros to a multiple of 8 NT): thread t owns the positions
// [8 q t, 8 q (t + 1)), q = ceil(len / 8NT).
template <int NT>
__device__ void compact_flags(const uint8_t* flags, int len, uint32_t* wave_sum, uint32_t* sel, int top_k,
                              uint32_t* total_out) {
  const int tid = threadIdx.x;
  const int q = (len + 8 * NT - 1) / (8 * NT);
  const uint64_t* mine = reinterpret_cast<const uint64_t*>(flags) + tid * q;
  uint32_t cnt = 0;
  for (int i = 0; i < q; ++i) cnt += __popcll(mine[i]);
  uint32_t total = 0;
  uint32_t at = block_exclusive_scan<NT>(wave_sum, cnt, &total);
  __syncthreads();  // sel may alias buffers read before this call
  for (int i = 0; i < q; ++i) {
    uint64_t bits = mine[i];
    while (bits) {
      const int bit = __ffsll((unsigned long long)bits) - 1;
      bits &= bits - 1;
      if (at < (uint32_t)top_k) sel[at] = (uint32_t)(8 * (tid * q + i) + (bit >> 3));
      ++at;
    }
  }
  __syncthreads();
  *total_out = total;
}

struct RowOut {
  int32_t* page;       // page-translated output (or the untranslated output)
  int32_t* raw;        // optional raw positions
  const int32_t* pt;   // page table row (NULL: write positions + offset)
  uint32_t page_bits;
  int32_t offset;      // ragged offset
  __device__ __forceinline__ void emit(int slot, int32_t p) const {
    if (pt) {
      int32_t v = -1;
      if (p >= 0) {
        const uint32_t mask = (1u << page_bits) - 1u;
        v = (pt[(uint32_t)p >> page_bits] << page_bits) | ((uint32_t)p & mask);
      }
      page[slot] = v;
      if (raw) raw[slot] = p;
    } else {
      page[slot] = p >= 0 ? p + offset : -1;
    }
  }
};

struct RowIn {
  const float* scores;
  int64_t stride;
  const int32_t* seq_lens;
  const int32_t* row_starts;
  int64_t max_len;
  // 1: scores that are not finite or have |x| >= 1e30 rank as -inf (the
  // portable selection tail of the indexer, lightning.py:1474-1478); 0: only
  // NaN does (topk_transform, topk.cuh).
  int mask_extreme;
  __device__ __forceinline__ uint32_t key(float x) const {
    return order_key(mask_extreme && !(fabsf(x) < 1e30f) ? -__builtin_inff() : x);
  }
  __device__ __forceinline__ int len(int b) const {
    int64_t l = seq_lens[b];
    return (int)(l < 0 ? 0 : (l > max_len ? max_len : l));
  }
  __device__ __forceinline__ const float* row(int b) const {
    return scores + (int64_t)b * stride + (row_starts ? row_starts[b] : 0);
  }
};

// ---------------------------------------------------------------- 1. threshold
__global__ void __launch_bounds__(kAuxThreads)
topk_threshold_kernel(const RowIn in, int top_k, RowWs* __restrict__ ws) {
  __shared__ __align__(16) uint32_t hist[kHistBins];
  __shared__ uint32_t wave_sum[kAuxThreads / 64];
  __shared__ uint32_t tb, above, eq;
  const int tid = threadIdx.x, b = blockIdx.x;
  const int len = in.len(b);
  RowWs& w = ws[b];
  if (len <= top_k) {
    if (tid == 0) { w.t_key = 0u; w.count = 0u; w.failed = 0u; }
    return;
  }
  const float* row = in.row(b);
  for (int i = tid; i < kHistBins; i += kAuxThreads) hist[i] = 0u;
  __syncthreads();
  // sampled chunks start at multiples of kSampleChunk * kSampleEvery
  constexpr int kStride = kSampleChunk * kSampleEvery;
  const int nchunks = (len + kStride - 1) / kStride;
  for (int c0 = 0; c0 < nchunks; c0 += 8) {
    float x[8][4];
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int pos = (c0 + c) * kStride + e * kAuxThreads + tid;
        x[c][e] = (c0 + c < nchunks && pos < len) ? row[pos] : 0.f;
      }
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int pos = (c0 + c) * kStride + e * kAuxThreads + tid;
        if (c0 + c < nchunks && pos < len) atomicAdd(&hist[in.key(x[c][e]) >> 20], 1u);
      }
  }
  uint32_t nsample = 0;
  for (int c = 0; c < nchunks; ++c) nsample += (uint32_t)max(0, min(len - c * kStride, kSampleChunk));
  const float fk = (float)nsample / (float)len * (float)top_k;
  const uint32_t r = (uint32_t)(fk + 4.f * sqrtf(fk) + 8.f);
  __syncthreads();
  uint32_t t_key = 0u;  // 0: gather everything
  if (r < nsample) {
    find_threshold<kAuxThreads>(hist, wave_sum, 4096, r, &tb, &above, &eq);
    const uint32_t tb0 = tb, rem0 = r - above;
    __syncthreads();
    for (int i = tid; i < 1024; i += kAuxThreads) hist[i] = 0u;
    __syncthreads();
    for (int c = 0; c < nchunks; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int pos = c * kStride + e * kAuxThreads + tid;
        if (pos < len) {
          const uint32_t k = in.key(row[pos]);  // second look at the sample: L2 hits
          if ((k >> 20) == tb0) atomicAdd(&hist[(k >> 10) & 1023u], 1u);
        }
      }
    __syncthreads();
    find_threshold<kAuxThreads>(hist, wave_sum, 1024, rem0, &tb, &above, &eq);
    t_key = (tb0 << 20) | (tb << 10);
  }
  if (tid == 0) {
    w.t_key = t_key;
    w.count = 0u;
    w.failed = 0u;
  }
}

// ---------------------------------------------------------------- 2. gather
__global__ void __launch_bounds__(kAuxThreads)
topk_gather_kernel(const RowIn in, int top_k, RowWs* __restrict__ ws) {
  __shared__ uint32_t s_key[kGatherLdsCap];
  __shared__ uint32_t s_pos[kGatherLdsCap];
  __shared__ uint32_t s_count, s_base;
  const int tid = threadIdx.x, lane = tid & 63, b = blockIdx.y;
  const int len = in.len(b);
  const int span0 = blockIdx.x * kGatherSpan;
  if (len <= top_k || span0 >= len) return;
  const float* row = in.row(b);
  RowWs& w = ws[b];
  if (tid == 0) s_count = 0u;
  const uint32_t t_key = w.t_key;
  // -inf and NaN share the lowest key; at or below it every element is gathered
  const bool all = t_key <= order_key(-__builtin_inff());
  const float t_f = key_to_float(t_key);
  float x[kGatherPerThread];
#pragma unroll
  for (int j = 0; j < kGatherPerThread; ++j) {
    const int pos = span0 + j * kAuxThreads + tid;
    x[j] = pos < len ? __builtin_nontemporal_load(row + pos) : 0.f;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kGatherPerThread; ++j) {
    const int pos = span0 + j * kAuxThreads + tid;
    // the float compare admits every key >= t_key (and -0.0 against +0.0,
    // which only adds a candidate)
    const bool pred = pos < len && (all || x[j] >= t_f);
    const uint64_t m = __ballot(pred);
    if (m) {
      const int leader = __builtin_ctzll(m);
      uint32_t base = 0;
      if (lane == leader) base = atomicAdd(&s_count, (uint32_t)__popcll(m));
      base = __shfl(base, leader, 64);
      if (pred) {
        const uint32_t slot = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        if (slot < kGatherLdsCap) {
          s_key[slot] = in.key(x[j]);
          s_pos[slot] = (uint32_t)pos;
        }
      }
    }
  }
  __syncthreads();
  const uint32_t n = s_count;
  if (tid == 0) {
    // an overflowing workgroup poisons the count so that the row falls back
    s_base = n ? atomicAdd(&w.count, n > kGatherLdsCap ? (uint32_t)(kListCap + 1) : n) : 0u;
  }
  __syncthreads();
  const uint32_t base = s_base;
  if (n <= kGatherLdsCap)
    for (uint32_t e = tid; e < n; e += kAuxThreads)
      if (base + e < kListCap) {
        w.key[base + e] = s_key[e];
        w.pos[base + e] = s_pos[e];
      }
}

// ---------------------------------------------------------------- 3. finish
// The finish of row b by one workgroup of kTopkThreads threads (all of them
// call it): the list select when the row's list is usable, else the full
// exact select over the row's scores.
__device__ __forceinline__ void finish_row(TopkSmem& s, const RowIn& in, RowWs* __restrict__ ws, const int32_t* __restrict__ offsets,
                           const int32_t* __restrict__ page_table, int64_t pt_stride, int pt_div, uint32_t page_bits,
                           int32_t* __restrict__ out_page, int32_t* __restrict__ out_raw, int top_k, int b) {
  const int tid = threadIdx.x;
  const int len = in.len(b);
  const float* row = in.row(b);

  RowOut out;
  out.page = out_page + (int64_t)b * top_k;
  out.raw = out_raw ? out_raw + (int64_t)b * top_k : nullptr;
  out.pt = page_table ? page_table + (int64_t)(b / pt_div) * pt_stride : nullptr;
  out.page_bits = page_bits;
  out.offset = offsets ? offsets[b] : 0;

  if (len <= top_k) {
    for (int i = tid; i < top_k; i += kTopkThreads) out.emit(i, i < len ? i : -1);
    return;
  }

  const int nwords = (len + 31) >> 5;
  for (int i = tid; i < nwords; i += kTopkThreads) s.bitmap[i] = 0u;
  for (int i = tid; i < kHistBins; i += kTopkThreads) s.hist[i] = 0u;
  if (tid < 2) s.list_count[tid] = 0u;
  const uint32_t cand = ws ? ws[b].count : 0u;
  const bool listed = ws && cand >= (uint32_t)top_k && cand <= (uint32_t)kListCap;
  __syncthreads();

  uint32_t thr[kLevels] = {0, 0, 0, 0, 0};
  uint32_t remain = (uint32_t)top_k;
  bool source_mode = !listed;  // level pass over the row (HBM) vs the LDS list
  int cur = 0;
  uint32_t list_n = 0;

  if (listed) {
    for (uint32_t e = tid; e < cand; e += kTopkThreads) {
      const uint32_t key = ws[b].key[e];
      s.list_key[0][e] = key;
      s.list_pos[0][e] = ws[b].pos[e];
      atomicAdd(&s.hist[key >> 20], 1u);
    }
    list_n = cand;
  } else {
    // Level-0 histogram: one coalesced pass over the row, 4 loads in flight per thread.
    for (int base = 0; base < len; base += 4 * kTopkThreads) {
      float x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = base + j * kTopkThreads + tid;
        x[j] = i < len ? row[i] : 0.f;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = base + j * kTopkThreads + tid;
        if (i < len) atomicAdd(&s.hist[in.key(x[j]) >> 20], 1u);
      }
    }
  }
  __syncthreads();

  for (int level = 0; level < kLevels; ++level) {
    find_threshold<kTopkThreads>(s.hist, s.wave_sum, radix_bins(level), remain, &s.tb, &s.above, &s.eq);
    const uint32_t tb = s.tb, above = s.above, eq = s.eq;
    thr[level] = tb;
    remain -= above;
    const bool take_all = (eq == remain) || level == kLevels - 1;
    const bool collect = !take_all && (!source_mode || eq <= (uint32_t)kListCap);
    const int nxt = cur ^ 1;
    __syncthreads();  // everyone has read tb/above/eq and the old histogram
    if (!take_all) {
      for (int i = tid; i < radix_bins(level + 1); i += kTopkThreads) s.hist[i] = 0u;
      if (tid == 0) s.list_count[nxt] = 0u;
    }
    __syncthreads();

    // one element of the current bucket: mark, or pass on to the next digit
    auto visit = [&](uint32_t key, uint32_t pos) {
      const uint32_t d = radix_digit(level, key, pos);
      if (d > tb || (take_all && d == tb)) atomicOr(&s.bitmap[pos >> 5], 1u << (pos & 31));
      if (!take_all && d == tb) {
        atomicAdd(&s.hist[radix_digit(level + 1, key, pos)], 1u);
        if (collect) {
          const uint32_t slot = atomicAdd(&s.list_count[nxt], 1u);
          s.list_key[nxt][slot] = key;
          s.list_pos[nxt][slot] = pos;
        }
      }
    };

    if (source_mode) {
      // HBM pass over the row (the exact path with no bound)
      for (int base = 0; base < len; base += 4 * kTopkThreads) {
        float x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int i = base + j * kTopkThreads + tid;
          x[j] = i < len ? row[i] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int i = base + j * kTopkThreads + tid;
          const uint32_t key = in.key(x[j]);
          if (i < len && in_bucket(level, key, (uint32_t)i, thr)) visit(key, (uint32_t)i);
        }
      }
    } else {
      for (uint32_t e = tid; e < list_n; e += kTopkThreads) visit(s.list_key[cur][e], s.list_pos[cur][e]);
    }
    __syncthreads();
    if (take_all) break;
    if (collect) {
      source_mode = false;
      cur = nxt;
      list_n = s.list_count[cur];
    }
  }

  // Compact the bitmap in position order: positions in ascending order into
  // LDS, then the page-table translation as independent loads spread over all
  // threads
  uint32_t* sel = s.list_pos[0];
  uint32_t total = 0;
  compact_bitmap<kTopkThreads>(s.bitmap, nwords, s.wave_sum, sel, top_k, &total);
  for (int i = tid; i < top_k; i += kTopkThreads) out.emit(i, i < (int)total ? (int32_t)sel[i] : -1);
}

__global__ void __launch_bounds__(kTopkThreads)
topk_finish_kernel(const RowIn in, RowWs* __restrict__ ws, const int32_t* __restrict__ offsets,
                   const int32_t* __restrict__ page_table, int64_t pt_stride, int pt_div, uint32_t page_bits,
                   int32_t* __restrict__ out_page, int32_t* __restrict__ out_raw, int top_k) {
  extern __shared__ __align__(16) uint8_t smem_raw[];
  finish_row(*reinterpret_cast<TopkSmem*>(smem_raw), in, ws, offsets, page_table, pt_stride, pt_div, page_bits,
             out_page, out_raw, top_k, blockIdx.x);
}

// ---------------------------------------------------------------- row repair
// Full indexer logits of one row by the calling workgroup (kTopkThreads
// threads): wave w computes pages w, w + 8, ... of the row through three
// rotating page buffers, logits[t] for t < len.
__device__ void repair_row_logits(const RowRepair& rp, const int32_t* __restrict__ bt_row, int row, int len) {
  constexpr int kWaves = kTopkThreads / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v8i qa[1][4];
  float w[1][4][4];
  load_query(rp.q + (int64_t)row * kIdxHeads * kIdxHeadDim, rp.weights + (int64_t)row * kIdxHeads, lane, qa[0],
             w[0]);
  float* out = rp.logits + (int64_t)row * rp.logits_stride;
  const int npages = (len + kIdxPageTokens - 1) / kIdxPageTokens;
  const int n = npages > wave ? (npages - wave + kWaves - 1) / kWaves : 0;  // this wave's pages
  auto page_ptr = [&](int i) { return rp.kv + (int64_t)bt_row[wave + kWaves * i] * kIdxPageBytes; };
  auto compute = [&](const PageRegs& pr, int i) {
    const float v = page_head_sum<1>(pr, 0, lane, qa, w);
    const int t = (wave + kWaves * i) * kIdxPageTokens + lane;
    if (t < len) out[t] = v * pr.scale;
  };
  PageRegs buf0, buf1, buf2;
  if (0 < n) load_page(buf0, page_ptr(0), lane);
  if (1 < n) load_page(buf1, page_ptr(1), lane);
  for (int i = 0; i < n; i += 3) {
    if (i + 2 < n) load_page(buf2, page_ptr(i + 2), lane);
    compute(buf0, i);
    if (i + 3 < n) load_page(buf0, page_ptr(i + 3), lane);
    if (i + 1 < n) compute(buf1, i + 1);
    if (i + 4 < n) load_page(buf1, page_ptr(i + 4), lane);
    if (i + 2 < n) compute(buf2, i + 2);
  }
}

// ---------------------------------------------------------------- list select
// Exact top-k of a row's candidate list (fused indexer path), ranked by
// (score, lower position), one row per workgroup. The first digit is a bin of
// the score (ListBins); the threshold bin's few candidates count those ahead of
// them. A crowded bin is binned again over its own range, and ties take radix
// levels, each a pass over the list: no usable list is redone from the logits,
// however its scores lie. (Radix digits of the key's bits, all levels, took 17.0
// us for four rows of 4K tokens, whose scores cross zero: sign and exponent bits
// put most candidates into a few bins, where the LDS atomics serialise. Bins
// linear in the score between the list's extremes: 128 rows of 64K, normal
// scores 14.0 us here and there, one outlier in each 26.8 against 15.3; 16 rows
// of 128K with a long tail 716 against 15.0, as a crowded bin of more than 6144
// made the row be redone.)
// kRepair: a row whose list is unusable (fewer than k entries, or more than its
// capacity) is redone in the kernel from its full logits (rp.q set, the launch
// reserves TopkSmem); otherwise it is appended to rp.defer_rows.
template <bool kRepair, typename RowList>
__device__ __forceinline__ void list_select_row(const int32_t* __restrict__ seq_lens, int64_t max_len,
                                                RowList* __restrict__ ws, const int32_t* __restrict__ page_table,
                                                int64_t pt_stride, int pt_div, uint32_t page_bits,
                                                const int32_t* __restrict__ offsets, int32_t* __restrict__ out_page,
                                                int32_t* __restrict__ out_raw, int top_k, const RowRepair& rp) {
  extern __shared__ __align__(16) uint8_t smem_raw[];
  ListSmem& s = *reinterpret_cast<ListSmem*>(smem_raw);
  constexpr int NT = kTopkThreads;
  const int tid = threadIdx.x, lane = tid & 63;
  const int b = blockIdx.x;
  const int64_t l = seq_lens[b];
  const int len = (int)(l < 0 ? 0 : (l > max_len ? max_len : l));
  RowList& w = ws[b];

  RowOut out;
  out.page = out_page + (int64_t)b * top_k;
  out.raw = out_raw ? out_raw + (int64_t)b * top_k : nullptr;
  out.pt = page_table ? page_table + (int64_t)(b / pt_div) * pt_stride : nullptr;
  out.page_bits = page_bits;
  out.offset = (!page_table && offsets) ? offsets[b] : 0;

  if (len <= top_k) {
    for (int i = tid; i < top_k; i += NT) out.emit(i, i < len ? i : -1);
    return;
  }
  const uint32_t cand = __builtin_amdgcn_readfirstlane(w.count);
  const auto select_list = [&]() {
  // The first kReg * NT candidates into registers (element e = u * NT + tid),
  // all loads in flight at once; any beyond them (a misjudged threshold) are
  // read again by each pass. Slots past the list are skipped by uniform
  // branches (most lists fill two thirds of the registers).
  constexpr int kReg = 12;
  uint32_t ch[kReg], cl[kReg];
#pragma unroll
  for (int u = 0; u < kReg; ++u) {
    const uint32_t e = (uint32_t)(u * NT + tid);
    ch[u] = 0u;
    cl[u] = 0u;
    if (e < cand) {
      ch[u] = w.key[e];
      cl[u] = w.pos[e];
    }
  }
  uint32_t cd[kReg];  // their bins
  // f(key, position, bin) over this thread's candidates; the bin is kept where it
  // is in registers, and otherwise made again by bin_of(key)
  auto each = [&](auto&& bin_of, auto&& f) {
#pragma unroll
    for (int u = 0; u < kReg; ++u)
      if ((uint32_t)(u * NT) < cand && (uint32_t)(u * NT + tid) < cand) f(ch[u], cl[u], cd[u]);
    for (uint32_t e = kReg * NT + tid; e < cand; e += NT) {
      const uint32_t key = w.key[e];
      uint32_t d = bin_of(key);
      f(key, w.pos[e], d);
    }
  };
  // The selected positions are marked in LDS: a byte each where the row fits
  // (plain stores), else a bit each. In a short row most positions are
  // selected and the lanes of a wave hold consecutive ones, so that atomics on
  // the bits serialise: 16.5 us against 11.5 for four rows of 1K to 4K tokens.
  const int npg = out.pt ? (len + (1 << page_bits) - 1) >> page_bits : 0;
  const int flag_words = (len + 8 * NT - 1) / (8 * NT) * (2 * NT);
  const bool bytes = flag_words + npg <= kBitmapWords;
  const int nwords = bytes ? flag_words : (len + 31) >> 5;
  // The row's page table, when it fits in the words past the marks, is copied
  // to LDS with the candidates so that the output's translation reads LDS, not
  // a dependent global load.
  const int pt_off = (nwords + 3) & ~3;
  const bool pt_lds = out.pt && pt_off + npg <= kBitmapWords;
  int32_t* const ptc = reinterpret_cast<int32_t*>(s.bitmap + pt_off);
  if (pt_lds) {
    for (int i0 = 0; i0 < npg; i0 += 4 * NT) {
      int32_t v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + u * NT + tid;
        v[u] = i < npg ? out.pt[i] : 0;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + u * NT + tid;
        if (i < npg) ptc[i] = v[u];
      }
    }
  }
  for (int i = tid; i < nwords; i += NT) s.bitmap[i] = 0u;
  for (int i = tid; i < kHistBins; i += NT) s.hist[i] = 0u;
  if (tid == 0) s.count = 0u;
  // the range of the scores above -inf (which ranks below every bin's start)
  const uint32_t ninf = order_key(-__builtin_inff()), fmax_key = order_key(3.4028235e38f);
  uint32_t kmin = 0xffffffffu, kmax = 0u;
  each([](uint32_t) { return 0u; }, [&](uint32_t key, uint32_t, uint32_t&) {
    kmin = min(kmin, key > ninf ? key : 0xffffffffu);
    kmax = max(kmax, key);
  });
  const uint32_t wave_top = block_range<NT>(s.wave_sum, kmin, kmax);
  uint8_t* const flags = reinterpret_cast<uint8_t*>(s.bitmap);
  auto mark = [&](uint32_t pos) {
    if (bytes) flags[pos] = 1;
    else atomicOr(&s.bitmap[pos >> 5], 1u << (pos & 31));
  };

  // First digit, straight from the registers. Bin 0 is counted in registers: a
  // crowd in it would serialise on one LDS word. Bins linear in the score end at
  // the lowest of the waves' largest scores: a few outliers share the last bin
  // with the few scores above that, far from the border.
  const ListBins bins(kmin, min(kmax, fmax_key), min(wave_top, fmax_key));
  uint32_t remain = (uint32_t)top_k;
  uint32_t lowest = 0;
  each([](uint32_t) { return 0u; }, [&](uint32_t key, uint32_t, uint32_t& d) {
    d = bins.of(key);
    if (d) atomicAdd(&s.hist[d], 1u);
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
  // Candidates in a higher bin are selected; the threshold bin's are ranked if
  // they are few, or their range is taken (bins never decrease with the key, so
  // that it holds no others).
  uint32_t low = 0xffffffffu, high = 0u;
  each([&](uint32_t key) { return bins.of(key); }, [&](uint32_t key, uint32_t pos, uint32_t d) {
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
  if (ranked) {
    // each of the threshold bin's candidates counts those ahead of it
    if ((uint32_t)tid < eq) {
      const uint64_t mine = s.rank[tid];
      uint32_t ahead = 0;
      for (uint32_t j = 0; j < eq; ++j) ahead += s.rank[j] > mine ? 1u : 0u;
      if (ahead < remain) mark(kIdxMax - (uint32_t)(mine & kIdxMax));
    }
  } else if (!whole_bin) {
    // A crowded bin reads the list again (from L2, four entries in flight), so
    // that it costs the usual case no registers.
    block_range<NT>(s.wave_sum, low, high);
    auto again = [&](auto&& f) {
#pragma unroll 1
      for (uint32_t e0 = tid; e0 < cand; e0 += 4 * NT) {
        uint32_t key[4], pos[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const uint32_t e = e0 + u * NT;
          key[u] = e < cand ? w.key[e] : 0u;
          pos[u] = e < cand ? w.pos[e] : 0u;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (e0 + u * NT < cand) f(key[u], pos[u]);
      }
    };
    select_crowd<NT, ListBins>(s, low, high, remain, again, mark, [](uint32_t, uint32_t) { return false; });
  }

  // compaction in position order and output
  __syncthreads();  // every mark is set
  uint32_t* sel = s.hist;  // 4096 entries >= top_k
  uint32_t total = 0;
  if (bytes) compact_flags<NT>(flags, len, s.wave_sum, sel, top_k, &total);
  else compact_bitmap<NT>(s.bitmap, nwords, s.wave_sum, sel, top_k, &total);
  if (pt_lds) {
    const uint32_t mask = (1u << page_bits) - 1u;
    for (int i = tid; i < top_k; i += NT) {
      const int32_t p = i < (int)total ? (int32_t)sel[i] : -1;
      out.page[i] = p >= 0 ? (int32_t)(((uint32_t)ptc[(uint32_t)p >> page_bits] << page_bits) | ((uint32_t)p & mask)) : -1;
      if (out.raw) out.raw[i] = p;
    }
  } else {
    for (int i = tid; i < top_k; i += NT) out.emit(i, i < (int)total ? (int32_t)sel[i] : -1);
  }
  };
  if (cand >= (uint32_t)top_k && cand <= (uint32_t)RowList::kCap) {
    select_list();
    return;
  }

  // A row whose list cannot give the exact top-k (the sample misjudged its
  // threshold) is redone here, from its full logits, or left to the caller.
  if (tid == 0) w.failed = 1u;
  if constexpr (kRepair) {
    repair_row_logits(rp, page_table + (int64_t)(b / pt_div) * pt_stride, b, len);
    __syncthreads();  // the row's logits (global) are visible to the whole workgroup
    const RowIn in{rp.logits, rp.logits_stride, seq_lens, nullptr, max_len};
    // a repairing launch reserves the full select's LDS
    finish_row(*reinterpret_cast<TopkSmem*>(smem_raw), in, nullptr, nullptr, page_table, pt_stride, pt_div,
               page_bits, out_page, out_raw, top_k, b);
  } else {
    if (tid == 0) rp.defer_rows[atomicAdd(rp.defer_count, 1u)] = b;
  }
}

__global__ void __launch_bounds__(kTopkThreads)
topk_list_kernel(const int32_t* __restrict__ seq_lens, int64_t max_len, DecodeList* __restrict__ ws,
                 const int32_t* __restrict__ page_table, int64_t pt_stride, int pt_div, uint32_t page_bits,
                 int32_t* __restrict__ out_page, int32_t* __restrict__ out_raw, int top_k, const RowRepair rp) {
  list_select_row<true, DecodeList>(seq_lens, max_len, ws, page_table, pt_stride, pt_div, page_bits, nullptr, out_page,
                                    out_raw, top_k, rp);
}

// Four waves per SIMD (<= 128 VGPRs): with the list layout, two workgroups per CU.
__global__ void __launch_bounds__(kTopkThreads) __attribute__((amdgpu_waves_per_eu(4)))
topk_list_defer_kernel(const int32_t* __restrict__ seq_lens, int64_t max_len, PrefillList* __restrict__ ws,
                       const int32_t* __restrict__ offsets, int32_t* __restrict__ out, int top_k,
                       const RowRepair rp) {
  list_select_row<false, PrefillList>(seq_lens, max_len, ws, nullptr, 0, 1, 0u, offsets, out, nullptr, top_k, rp);
}

// ---------------------------------------------------------------- row select
// Exact top-k of a row of up to 64K scores by one workgroup, which reads the
// row once: thread t holds positions [4t, 4t + 4) of every chunk of 4096 in
// registers. First digit: the score's bin (linear in its bits or in the score),
// counted over the whole row; the threshold bin's few elements count those ahead
// of them, a crowded bin is binned again, and ties are numbered by position. The
// selected positions are a bitmap in LDS, compacted in position order by one
// block scan.
//
// What bounds it: a chain of short phases in one CU (loads, extremes, LDS
// histogram, threshold, ranks, compaction). A 1/8 sample's threshold, the
// candidates above it listed and three radix levels over the list took
// 31 us a call for 33 rows of 40000 scores where this takes 20.3, for normal
// scores as for ones with an outlier or a long tail, and 153 for four distinct
// scores where this takes 61. (Bins linear in the score alone: 17.4 for normal
// scores, but 91 with one outlier of 1e9.)
// Instantiated per power of two of the row's chunks: a kernel for longer rows
// spends its registers and tests on chunks that a short one does not have.
constexpr int kRowThreads = 1024;
constexpr int kRowChunk = 4 * kRowThreads;
constexpr int kRowMaxChunks = kRowSelectLen / kRowChunk;
static_assert(kRowMaxChunks == 16, "the largest instantiation");
struct RowSelectSmem {
  uint32_t hist[kHistBins];  // then the selected positions
  uint64_t rank[kRankCap];
  uint32_t bits[kRowSelectLen / 32];
  uint32_t wave_sum[2 * (kRowThreads / 64)];
  float floors[kRowThreads / 64];
  uint32_t count, tb, above, eq;
};

// Bitwise or over each group of 8 lanes.
__device__ __forceinline__ uint32_t or_8_lanes(uint32_t x) {
  x |= (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xb1, 0xf, 0xf, true);   // lane ^ 1
  x |= (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4e, 0xf, 0xf, true);   // lane ^ 2
  x |= (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x141, 0xf, 0xf, true);  // lane ^ 7: the other four
  return x;
}

template <int kChunks>
__global__ void __launch_bounds__(kRowThreads)
topk_row_kernel(const RowIn in, const int32_t* __restrict__ offsets, const int32_t* __restrict__ page_table,
                int64_t pt_stride, int pt_div, uint32_t page_bits, int32_t* __restrict__ out_page,
                int32_t* __restrict__ out_raw, int top_k) {
  __shared__ __align__(16) RowSelectSmem s;
  constexpr int NT = kRowThreads, NW = NT / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int b = blockIdx.x;
  const int len = in.len(b);
  const RowOut out{out_page + (int64_t)b * top_k, out_raw ? out_raw + (int64_t)b * top_k : nullptr,
                   page_table ? page_table + (int64_t)(b / pt_div) * pt_stride : nullptr, page_bits,
                   offsets ? offsets[b] : 0};
  if (len <= top_k) {
    for (int i = tid; i < top_k; i += NT) out.emit(i, i < len ? i : -1);
    return;
  }
  const float* row = in.row(b);
  const int nch = (len + kRowChunk - 1) / kRowChunk;
  const float inf = __builtin_inff();

  // ---- the row. The launcher guarantees 16-byte aligned rows; a quad that
  // would pass the row's storage reads the last whole quad instead, so no load
  // sits behind a lane's branch, and the storage's last max_len % 4 scores are
  // read one by one. Positions at or past the length hold -inf: they rank
  // behind all len > top_k real elements, so they are never selected.
  const int last = (int)((in.max_len - 4) & ~(int64_t)3);
  float x[4 * kChunks];
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    v4f v = {-inf, -inf, -inf, -inf};
    if (c < nch) v = *reinterpret_cast<const v4f*>(row + min(kRowChunk * c + 4 * tid, last));
#pragma unroll
    for (int e = 0; e < 4; ++e) x[4 * c + e] = v[e];
  }
  for (int i = tid; i < kHistBins; i += NT) s.hist[i] = 0u;
  if (tid == 0) s.count = 0u;
  // scores that rank as -inf: NaN, and for the indexer's tail |x| >= 1e30
  const float cap = in.mask_extreme ? __uint_as_float(__float_as_uint(1e30f) - 1u) : inf;
  auto score = [&](int p, int e, float v) {  // v: what was read for position p + e
    if (p > last) v = p + e < len ? row[p + e] : -inf;
    return p + e < len && fabsf(v) <= cap ? v : -inf;
  };
  float lo = inf, hi = -inf;  // the extremes; lo of the scores above -inf
  float second = -inf;        // this thread's second highest
#pragma unroll
  for (int c = 0; c < kChunks; ++c)
    if (c < nch) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float& v = x[4 * c + e];
        v = score(kRowChunk * c + 4 * tid, e, v);
        lo = fminf(lo, v > -inf ? v : inf);
        second = fmaxf(second, fminf(hi, v));
        hi = fmaxf(hi, v);
      }
    }
  auto block_extremes = [&](float& low, float& high) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      low = fminf(low, __shfl_xor(low, off, 64));
      high = fmaxf(high, __shfl_xor(high, off, 64));
    }
    float* wave_f = reinterpret_cast<float*>(s.wave_sum);
    if (lane == 0) {
      wave_f[wave] = low;
      wave_f[NW + wave] = high;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      low = fminf(low, wave_f[i]);
      high = fmaxf(high, wave_f[NW + i]);
    }
  };
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) second = fminf(second, __shfl_xor(second, off, 64));
  if (lane == 0) s.floors[wave] = second;
  block_extremes(lo, hi);
#pragma unroll
  for (int i = 0; i < NW; ++i) second = fminf(second, s.floors[i]);
  uint32_t remain = (uint32_t)top_k;
  uint32_t crowd_low = 0u, crowd_high = 0u;  // the keys of a threshold bin too crowded to rank
  auto decide = [&](const auto bins) {

  // ---- first digit. Scores with a long tail (or many at the lowest value)
  // fill bin 0: it is counted in registers, where one LDS word would serialise.
  auto add_lowest = [&](uint32_t n) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) n += (uint32_t)__shfl_xor(n, off, 64);
    if (lane == 0 && n) atomicAdd(&s.hist[0], n);
  };
  uint32_t lowest = 0;
#pragma unroll
  for (int c = 0; c < kChunks; ++c)
    if (c < nch && kRowChunk * c + 4 * tid < len) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t d = bins.bin(x[4 * c + e]);
        if (d) atomicAdd(&s.hist[d], 1u);
        else ++lowest;
      }
    }
  add_lowest(lowest);
  __syncthreads();
  find_threshold<NT>(s.hist, s.wave_sum, kHistBins, remain, &s.tb, &s.above, &s.eq);
  const uint32_t tb = s.tb, eq = s.eq;
  remain -= s.above;
  const bool whole_bin = eq == remain;
  const uint32_t sure = whole_bin ? tb : tb + 1;  // bins selected whole
  const bool ranked = !whole_bin && eq <= (uint32_t)kRankCap;
  uint32_t low = 0xffffffffu, high = 0u;  // the keys of a crowded threshold bin
#pragma unroll
  for (int c = 0; c < kChunks; ++c)
    if (c < nch) {
      const int p = kRowChunk * c + 4 * tid;
      uint32_t quad = 0u;
      if (p < len) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t d = bins.bin(x[4 * c + e]);
          if (d >= sure) {
            quad |= 1u << e;
          } else if (d == tb) {
            const uint32_t key = order_key(x[4 * c + e]);
            if (ranked) {
              s.rank[atomicAdd(&s.count, 1u)] = rank_composite(key, (uint32_t)(p + e));
            } else {
              low = min(low, key);
              high = max(high, key);
            }
          }
        }
      }
      // eight lanes' quads are a word of the bitmap
      const uint32_t word = or_8_lanes(quad << (4 * (lane & 7)));
      if ((lane & 7) == 0) s.bits[p >> 5] = word;
    }
  __syncthreads();
  if (ranked) {
    // the threshold bin's elements: those with fewer than `remain` ahead of them
    if ((uint32_t)tid < eq) {
      const uint64_t mine = s.rank[tid];
      uint32_t ahead = 0;
      for (uint32_t e = 0; e < eq; ++e) ahead += s.rank[e] > mine ? 1u : 0u;
      const uint32_t pos = kIdxMax - (uint32_t)(mine & kIdxMax);
      if (ahead < remain) atomicOr(&s.bits[pos >> 5], 1u << (pos & 31));
    }
  } else if (!whole_bin) {
    // Too many elements for that. The row is read again (from L2, four chunks in
    // flight), so that this costs the usual case no registers.
    block_range<NT>(s.wave_sum, low, high);
    crowd_low = low;
    crowd_high = high;
  }
  return ranked || whole_bin;
  };
  // The 2 x 1024 scores that are some thread's highest two are at least `second`,
  // so that the top-k (at most 2048) is: above it the bins are linear in the
  // float's bits (outliers and long tails then cost a few octaves of bins, not
  // the range), unless it is negative (rows of a few scores per thread), where
  // that would spend the bins around zero. Infinities fall into the end bins.
  const float top = fminf(hi, 3.4028235e38f);
  const bool decided = second > 0.f ? decide(BitBins(second, top)) : decide(ScoreBins(lo, top));
  if (!decided) {
    auto quads = [&](auto&& visit) {  // visit(chunk, position, the quad's keys)
#pragma unroll 1
      for (int c0 = 0; c0 < nch; c0 += 4) {
        v4f v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (c0 + u < nch) v[u] = *reinterpret_cast<const v4f*>(row + min(kRowChunk * (c0 + u) + 4 * tid, last));
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int p = kRowChunk * (c0 + u) + 4 * tid;
          if (p >= len) continue;
          uint4 key;
          key.x = order_key(score(p, 0, v[u][0]));
          key.y = order_key(score(p, 1, v[u][1]));
          key.z = order_key(score(p, 2, v[u][2]));
          key.w = order_key(score(p, 3, v[u][3]));
          visit(c0 + u, p, key);
        }
      }
    };
    auto again = [&](auto&& visit) {
      quads([&](int, int p, const uint4& key) {
        visit(key.x, (uint32_t)p);
        visit(key.y, (uint32_t)(p + 1));
        visit(key.z, (uint32_t)(p + 2));
        visit(key.w, (uint32_t)(p + 3));
      });
    };
    auto mark = [&](uint32_t pos) { atomicOr(&s.bits[pos >> 5], 1u << (pos & 31)); };
    // One key's n lowest positions: positions rise with chunk, wave, lane and
    // quad element, so that counts per (chunk, wave) and one scan number them all
    // (33 rows of 40000 scores of ten values 37 us, all equal 33; by radix levels
    // from the first bin's range on, 85 and 74).
    auto ties = [&](uint32_t tie, uint32_t n) {
      uint64_t found = 0;  // four bits per chunk
      quads([&](int c, int p, const uint4& key) {
        const uint32_t m = (key.x == tie ? 1u : 0u) | (key.y == tie && p + 1 < len ? 2u : 0u) |
                           (key.z == tie && p + 2 < len ? 4u : 0u) | (key.w == tie && p + 3 < len ? 8u : 0u);
        found |= (uint64_t)m << (4 * c);
      });
      for (int c = 0; c < nch; ++c) {
        uint32_t in_wave = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) in_wave += (uint32_t)__popcll(__ballot((found >> (4 * c + e)) & 1ull));
        if (lane == 0) s.hist[c * NW + wave] = in_wave;
      }
      __syncthreads();
      uint32_t total = 0;
      const uint32_t before = block_exclusive_scan<NT>(s.wave_sum, tid < nch * NW ? s.hist[tid] : 0u, &total);
      if (tid < nch * NW) s.hist[tid] = before;
      __syncthreads();
      for (int c = 0; c < nch; ++c) {
        uint32_t at = s.hist[c * NW + wave];
        if (at >= n) break;
        const uint32_t mine = (uint32_t)(found >> (4 * c)) & 15u;
#pragma unroll
        for (int e = 0; e < 4; ++e) at += (uint32_t)__popcll(__ballot((mine >> e) & 1u) & ((1ull << lane) - 1ull));
        uint32_t quad = 0u;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if ((mine >> e) & 1u) {
            if (at < n) quad |= 1u << e;
            ++at;
          }
        const uint32_t word = or_8_lanes(quad << (4 * (lane & 7)));
        if ((lane & 7) == 0) s.bits[(kRowChunk * c + 4 * tid) >> 5] |= word;
      }
      return true;
    };
    select_crowd<NT, ScoreBins>(s, crowd_low, crowd_high, remain, again, mark, ties);
  }
  __syncthreads();

  // ---- positions in ascending order (thread t: `per` of them, a power of two,
  // at most two words), then the page translation
  int per = 4;
  while (per < 4 * nch) per *= 2;
  uint64_t mine = 0;
  if (tid * per < nch * kRowChunk) {
    const uint32_t* w = s.bits + ((tid * per) >> 5);
    mine = per == 64 ? w[0] | ((uint64_t)w[1] << 32) : (w[0] >> ((tid * per) & 31)) & (0xffffffffu >> (32 - per));
  }
  uint32_t total = 0;
  uint32_t at = block_exclusive_scan<NT>(s.wave_sum, (uint32_t)__popcll(mine), &total);
  __syncthreads();  // the histogram becomes the list of selected positions
  while (mine) {
    const int i = __ffsll((unsigned long long)mine) - 1;
    mine &= mine - 1;
    s.hist[at++] = (uint32_t)(tid * per + i);
  }
  __syncthreads();
  for (int i = tid; i < top_k; i += NT) out.emit(i, (int32_t)s.hist[i]);
}

static void launch_row(const RowIn& in, const int32_t* offsets, const int32_t* page_table, int64_t pt_stride,
                       int pt_div, uint32_t page_bits, int32_t* out_page, int32_t* out_raw, int top_k, int rows,
                       hipStream_t stream) {
  auto* kernel = in.max_len <= kRowChunk       ? topk_row_kernel<1>
                 : in.max_len <= 2 * kRowChunk ? topk_row_kernel<2>
                 : in.max_len <= 4 * kRowChunk ? topk_row_kernel<4>
                 : in.max_len <= 8 * kRowChunk ? topk_row_kernel<8>
                                               : topk_row_kernel<kRowMaxChunks>;
  hipLaunchKernelGGL(kernel, dim3(rows), dim3(kRowThreads), 0, stream, in, offsets, page_table, pt_stride, pt_div,
                     page_bits, out_page, out_raw, top_k);
}

__global__ void topk_to_physical_kernel(const int32_t* __restrict__ topk, int64_t topk_stride,
                                        const int32_t* __restrict__ bt, int64_t bt_stride,
                                        int table_width, int rows, int k, int rows_per_table,
                                        int block_size, int32_t* __restrict__ out) {
  const int64_t n = (int64_t)rows * k;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int r = (int)(e / k), c = (int)(e % k);
    const int32_t p = topk[(int64_t)r * topk_stride + c];
    int32_t v = -1;
    if (p >= 0) {
      const int page = p / block_size;
      if (page < table_width)
        v = bt[(int64_t)(r / rows_per_table) * bt_stride + page] * block_size + p % block_size;
    }
    out[e] = v;
  }
}

static int prepare_topk_kernel() {
  static int status = -1;
  if (status < 0) {
    hipError_t e = hipFuncSetAttribute((const void*)topk_finish_kernel,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTopkSmemBytes);
    if (e == hipSuccess)
      e = hipFuncSetAttribute((const void*)topk_list_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)kTopkSmemBytes);
    if (e == hipSuccess)
      e = hipFuncSetAttribute((const void*)topk_list_defer_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)sizeof(ListSmem));
    status = e == hipSuccess ? 0 : 1;
    if (status) return set_error(kLaunchFailed, "topk: cannot reserve %zu B of LDS: %s",
                                 kTopkSmemBytes, hipGetErrorString(e));
  }
  return status ? kLaunchFailed : kOk;
}

// The launches of one selection. `workspace` NULL: the exact full path only.
// Scratch of the no-allocation entry point: the per-row state (threshold,
// candidate count, candidate list) of up to kNoAllocRows rows, held by every
// GPU the library runs on until the process ends. Host code never passes the
// array's name to a kernel (on the host it is only a stand-in for the symbol):
// each device's address comes from hipGetSymbolAddress, once per device.
constexpr int kNoAllocRows = 256;
static __device__ __align__(256) uint8_t scratch[kNoAllocRows * sizeof(RowWs)];
constexpr int kMaxDevices = 64;
static void* g_scratch_ptr[kMaxDevices];
static std::mutex g_scratch_mu;

// This device's address of `scratch` (looked up on the first call with that
// device current, then cached).
static int device_scratch(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return set_error(kLaunchFailed, "dsa_topk_transform_noalloc: no usable current device (%d)", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return set_error(kLaunchFailed, "dsa_topk_transform_noalloc: hipGetSymbolAddress(scratch) failed: %s",
                       hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return kOk;
}

static int launch_topk(const RowIn& in, int batch, const int32_t* offsets, const int32_t* page_table,
                       int64_t pt_stride, uint32_t page_bits, int32_t* out_page, int32_t* out_raw,
                       int top_k, void* workspace, size_t workspace_bytes, hipStream_t stream,
                       const char* what) {
  if (int rc = prepare_topk_kernel()) return rc;
  const bool aligned = (reinterpret_cast<uintptr_t>(in.scores) & 15) == 0 && (in.stride & 3) == 0 && !in.row_starts;
  if (in.max_len <= kRowSelectLen && aligned) {
    // the whole row fits in one workgroup's registers: one launch, no workspace
    launch_row(in, offsets, page_table, pt_stride, 1, page_bits, out_page, out_raw, top_k, batch, stream);
    return check_launch(what);
  }
  RowWs* ws = nullptr;
  if (workspace) {
    if (workspace_bytes < (size_t)batch * sizeof(RowWs))
      return set_error(kWorkspaceTooSmall, "%s: workspace %zu B < %zu B", what, workspace_bytes,
                       (size_t)batch * sizeof(RowWs));
    if (reinterpret_cast<uintptr_t>(workspace) & 15)
      return set_error(kInvalidArgument, "%s: workspace must be 16-byte aligned", what);
    ws = static_cast<RowWs*>(workspace);
    hipLaunchKernelGGL(topk_threshold_kernel, dim3(batch), dim3(kAuxThreads), 0, stream, in, top_k, ws);
    const int64_t spans = (in.max_len + kGatherSpan - 1) / kGatherSpan;
    if (spans > 0)
      hipLaunchKernelGGL(topk_gather_kernel, dim3((unsigned)spans, batch), dim3(kAuxThreads), 0, stream, in,
                         top_k, ws);
  }
  hipLaunchKernelGGL(topk_finish_kernel, dim3(batch), dim3(kTopkThreads), kTopkSmemBytes, stream, in, ws,
                     offsets, page_table, pt_stride, 1, page_bits, out_page, out_raw, top_k);
  return check_launch(what);
}

int launch_list_select(const RowRepair& rp, const int32_t* seq_lens, int64_t max_len, DecodeList* ws,
                       const int32_t* page_table, int64_t pt_stride, int pt_div, uint32_t page_bits,
                       int32_t* out_page, int32_t* out_raw, int top_k, int rows, hipStream_t stream) {
  if (int rc = prepare_topk_kernel()) return rc;
  hipLaunchKernelGGL(topk_list_kernel, dim3(rows), dim3(kTopkThreads), kTopkSmemBytes, stream, seq_lens, max_len, ws,
                     page_table, pt_stride, pt_div, page_bits, out_page, out_raw, top_k, rp);
  return check_launch("dsa_indexer_topk(select)");
}

int launch_list_select(const RowRepair& rp, const int32_t* seq_lens, int64_t max_len, PrefillList* ws,
                       const int32_t* offsets, int32_t* out, int top_k, int rows, hipStream_t stream) {
  if (int rc = prepare_topk_kernel()) return rc;
  hipLaunchKernelGGL(topk_list_defer_kernel, dim3(rows), dim3(kTopkThreads), sizeof(ListSmem), stream, seq_lens,
                     max_len, ws, offsets, out, top_k, rp);
  return check_launch("dsa_mqa_topk(select)");
}

int launch_row_select(const float* scores, int64_t score_stride, const int32_t* seq_lens, int64_t max_len,
                      const int32_t* page_table, int64_t pt_stride, int pt_div, uint32_t page_bits, int32_t* out_page,
                      int32_t* out_raw, int top_k, int rows, hipStream_t stream) {
  const RowIn in{scores, score_stride, seq_lens, nullptr, max_len, 0};
  launch_row(in, nullptr, page_table, pt_stride, pt_div, page_bits, out_page, out_raw, top_k, rows, stream);
  return check_launch("dsa_indexer_topk(row select)");
}

}  // namespace dsa

extern "C" {

int dsa_topk_max_len(void) { return dsa::kTopkMaxLen; }

size_t dsa_topk_workspace_bytes(int batch) {
  return batch > 0 ? (size_t)batch * sizeof(dsa::RowWs) : 0;
}

int dsa_topk_transform(const float* scores, int64_t score_stride, const int32_t* seq_lens,
                       const int32_t* page_table, int64_t page_table_stride, int32_t* out_page,
                       int32_t* out_raw, int batch, int64_t max_len, int page_size, int top_k,
                       void* workspace, size_t workspace_bytes, void* stream) {
  using namespace dsa;
  if (top_k != 512 && top_k != 2048)
    return set_error(kInvalidArgument, "top_k must be 512 or 2048, got %d", top_k);
  if (page_size <= 0 || (page_size & (page_size - 1)))
    return set_error(kInvalidArgument, "page_size must be power of 2, got %d", page_size);
  if (batch < 0 || max_len < 0 || (batch > 0 && (!scores || !seq_lens || !out_page)))
    return set_error(kInvalidArgument, "dsa_topk_transform: bad arguments");
  if (max_len > kTopkMaxLen)
    return set_error(kUnsupported, "score rows longer than %d are not supported (got %lld)",
                     kTopkMaxLen, (long long)max_len);
  if (batch == 0) return kOk;
  const RowIn in{scores, score_stride, seq_lens, nullptr, max_len};
  const uint32_t bits = (uint32_t)__builtin_ctz((unsigned)page_size);
  return launch_topk(in, batch, nullptr, page_table, page_table_stride, bits, out_page,
                     page_table ? out_raw : nullptr, top_k, workspace, workspace_bytes, (hipStream_t)stream,
                     "dsa_topk_transform");
}

int dsa_topk_transform_noalloc(const float* scores, int64_t score_stride, const int32_t* seq_lens,
                               const int32_t* page_table, int64_t page_table_stride, int32_t* out_page,
                               int32_t* out_raw, int batch, int64_t max_len, int page_size, int top_k,
                               void* stream) {
  using namespace dsa;
  if (top_k != 512 && top_k != 2048)
    return set_error(kInvalidArgument, "top_k must be 512 or 2048, got %d", top_k);
  if (page_size <= 0 || (page_size & (page_size - 1)))
    return set_error(kInvalidArgument, "page_size must be power of 2, got %d", page_size);
  if (batch < 0 || max_len < 0 || (batch > 0 && (!scores || !seq_lens || !out_page)))
    return set_error(kInvalidArgument, "dsa_topk_transform_noalloc: bad arguments");
  if (batch > kNoAllocRows)
    return set_error(kUnsupported, "dsa_topk_transform_noalloc: %d rows exceed the scratch maximum of %d rows",
                     batch, kNoAllocRows);
  if (max_len > kTopkMaxLen)
    return set_error(kUnsupported, "score rows longer than %d are not supported (got %lld)",
                     kTopkMaxLen, (long long)max_len);
  if (batch == 0) return kOk;
  void* ws = nullptr;
  if (int rc = device_scratch(&ws)) return rc;
  const RowIn in{scores, score_stride, seq_lens, nullptr, max_len};
  const uint32_t bits = (uint32_t)__builtin_ctz((unsigned)page_size);
  return launch_topk(in, batch, nullptr, page_table, page_table_stride, bits, out_page,
                     page_table ? out_raw : nullptr, top_k, ws, (size_t)kNoAllocRows * sizeof(RowWs),
                     (hipStream_t)stream, "dsa_topk_transform_noalloc");
}

int dsa_indexer_select(const float* logits, int64_t logits_stride, const int32_t* context_lens,
                       int32_t* out, int rows, int64_t max_len, int top_k, void* workspace,
                       size_t workspace_bytes, void* stream) {
  using namespace dsa;
  if (top_k != 512 && top_k != 2048)
    return set_error(kInvalidArgument, "top_k must be 512 or 2048, got %d", top_k);
  if (rows < 0 || max_len < 0 || (rows > 0 && (!logits || !context_lens || !out)))
    return set_error(kInvalidArgument, "dsa_indexer_select: bad arguments");
  if (max_len > kTopkMaxLen)
    return set_error(kUnsupported, "logits rows longer than %d are not supported (got %lld)",
                     kTopkMaxLen, (long long)max_len);
  if (rows == 0) return kOk;
  const RowIn in{logits, logits_stride, context_lens, nullptr, max_len, 1};
  return launch_topk(in, rows, nullptr, nullptr, 0, 0u, out, nullptr, top_k, workspace, workspace_bytes,
                     (hipStream_t)stream, "dsa_indexer_select");
}

int dsa_topk_transform_ragged(const float* scores, int64_t score_stride, const int32_t* seq_lens,
                              const int32_t* row_starts, const int32_t* offsets, int32_t* out,
                              int batch, int64_t max_len, int top_k, void* workspace,
                              size_t workspace_bytes, void* stream) {
  using namespace dsa;
  if (top_k != 2048) return set_error(kInvalidArgument, "ragged Indexer top_k must be 2048, got %d", top_k);
  if (batch < 0 || max_len < 0 || (batch > 0 && (!scores || !seq_lens || !row_starts || !offsets || !out)))
    return set_error(kInvalidArgument, "dsa_topk_transform_ragged: bad arguments");
  if (max_len > kTopkMaxLen)
    return set_error(kUnsupported, "ragged rows longer than %d are not supported (got %lld)",
                     kTopkMaxLen, (long long)max_len);
  if (batch == 0) return kOk;
  const RowIn in{scores, score_stride, seq_lens, row_starts, max_len};
  return launch_topk(in, batch, offsets, nullptr, 0, 0u, out, nullptr, top_k, workspace, workspace_bytes,
                     (hipStream_t)stream, "dsa_topk_transform_ragged");
}

int dsa_topk_to_physical(const int32_t* topk_indices, int64_t topk_stride, const int32_t* block_table,
                         int64_t bt_stride, int table_width, int rows, int topk, int rows_per_table,
                         int block_size, int32_t* out, void* stream) {
  using namespace dsa;
  if (rows < 0 || topk < 0 || rows_per_table < 1 || block_size <= 0 || table_width < 0)
    return set_error(kInvalidArgument, "dsa_topk_to_physical: bad arguments");
  const int64_t n = (int64_t)rows * topk;
  if (n == 0) return kOk;
  if (!topk_indices || !block_table || !out)
    return set_error(kInvalidArgument, "dsa_topk_to_physical: null pointer");
  const int threads = 256;
  const int64_t blocks = std::min<int64_t>((n + threads - 1) / threads, 65536);
  hipLaunchKernelGGL(topk_to_physical_kernel, dim3((unsigned)blocks), dim3(threads), 0, (hipStream_t)stream,
                     topk_indices, topk_stride, block_table, bt_stride, table_width, rows, topk,
                     rows_per_table, block_size, out);
  return check_launch("dsa_topk_to_physical");
}

}  // extern "C"
