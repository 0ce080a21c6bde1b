// Sparse MLA prefill entry points, for gfx950: over ragged bf16 key rows, and
// over the paged fp8 cache plus the chunk's fresh bf16 rows. Both run the
// attention kernel of sparse_mla.hip; this file holds the split of a paged
// prefill's selected keys into cache slots and fresh rows.
#include "dsa_common.h"
#include "../../include/dsa_amd.h"

namespace dsa {
namespace {

// The chunked prefill's top-k split by where each key lives. Index g of token t
// is a position in the ragged key order (sequence b's keys at cu_k[b] ..): key
// i = g - cu_k[b] is cached row i of sequence b while i < k_len - q_len (its
// physical slot block_table[b][i / bs] * bs + i % bs in the paged fp8 cache),
// else fresh row cu_q[b] + i - (k_len - q_len). Each token's two lists are
// compacted in index order and padded with -1 to their widths, and their
// lengths go to counts[2t], counts[2t+1]. One 256-thread workgroup per token.
__global__ void __launch_bounds__(256)
prefill_split_kernel(const int32_t* __restrict__ idx, int64_t idx_stride, int topk, const void* __restrict__ cu_q,
                     const void* __restrict__ cu_k, int cu_is_64, int num_seqs, int64_t total_k,
                     const int32_t* __restrict__ bt, int64_t bt_stride, int bt_width, int block_size,
                     int32_t* __restrict__ cached, int cached_w, int32_t* __restrict__ fresh, int fresh_w,
                     int32_t* __restrict__ counts) {
  auto cu = [&](const void* p, int i) -> int64_t {
    return cu_is_64 ? reinterpret_cast<const int64_t*>(p)[i] : (int64_t)reinterpret_cast<const int32_t*>(p)[i];
  };
  __shared__ int s_cnt[2][4];
  __shared__ int s_base[2];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int32_t* row = idx + (int64_t)t * idx_stride;
  int32_t* crow = cached + (int64_t)t * cached_w;
  int32_t* frow = fresh + (int64_t)t * fresh_w;
  if (tid == 0) s_base[0] = s_base[1] = 0;
  for (int e0 = 0; e0 < topk; e0 += 256) {
    const int e = e0 + tid;
    int kind = -1;  // 0 cached, 1 fresh
    int32_t v = -1;
    const int64_t g = e < topk ? (int64_t)row[e] : -1;
    if (g >= 0 && g < total_k) {
      int lo = 0, hi = num_seqs;  // largest b < num_seqs with cu_k[b] <= g
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (cu(cu_k, mid) <= g) lo = mid; else hi = mid;
      }
      const int64_t k0 = cu(cu_k, lo), k1 = cu(cu_k, lo + 1);
      const int64_t ncached = (k1 - k0) - (cu(cu_q, lo + 1) - cu(cu_q, lo));
      const int64_t i = g - k0;
      if (i < ncached) {
        // a block-table column past the table's width is skipped like -1; a
        // stale or negative block gives a slot the MLA kernel skips
        const int64_t col = i / block_size;
        if (col < bt_width) {
          kind = 0;
          v = bt[(int64_t)lo * bt_stride + col] * block_size + (int32_t)(i % block_size);
        }
      } else {
        kind = 1;
        v = (int32_t)(cu(cu_q, lo) + i - ncached);
      }
    }
    const uint64_t mc = __ballot(kind == 0), mf = __ballot(kind == 1);
    if (lane == 0) {
      s_cnt[0][wave] = __popcll(mc);
      s_cnt[1][wave] = __popcll(mf);
    }
    __syncthreads();
    int bc = s_base[0], bf = s_base[1];
    for (int w = 0; w < wave; ++w) {
      bc += s_cnt[0][w];
      bf += s_cnt[1][w];
    }
    const uint64_t below = (1ull << lane) - 1ull;
    if (kind == 0) crow[bc + __popcll(mc & below)] = v;
    if (kind == 1) frow[bf + __popcll(mf & below)] = v;
    __syncthreads();
    if (tid == 0) {
      s_base[0] += s_cnt[0][0] + s_cnt[0][1] + s_cnt[0][2] + s_cnt[0][3];
      s_base[1] += s_cnt[1][0] + s_cnt[1][1] + s_cnt[1][2] + s_cnt[1][3];
    }
    __syncthreads();
  }
  const int nc = s_base[0], nf = s_base[1];
  if (tid == 0) {
    counts[2 * t] = nc;
    counts[2 * t + 1] = nf;
  }
  for (int e = nc + tid; e < cached_w; e += 256) crow[e] = -1;
  for (int e = nf + tid; e < fresh_w; e += 256) frow[e] = -1;
}

}  // namespace

static int sparse_mla_prefill_impl(const void* q, int64_t q_token_stride, int64_t q_head_stride, const void* kv,
                                   int64_t kv_row_stride, int64_t s_kv, const int32_t* indices, int64_t idx_stride,
                                   int num_tokens, int num_heads, int topk, float sm_scale, void* out,
                                   float* max_logits, float* lse, void* stream);
}  // namespace dsa

extern "C" {

int dsa_sparse_mla_prefill(const void* q, int64_t q_token_stride, int64_t q_head_stride, const void* kv,
                           int64_t kv_row_stride, int64_t s_kv, const int32_t* indices, int64_t idx_stride,
                           int num_tokens, int num_heads, int topk, float sm_scale, void* out, float* max_logits,
                           float* lse, void* stream) {
  return dsa::sparse_mla_prefill_impl(q, q_token_stride, q_head_stride, kv, kv_row_stride, s_kv, indices,
                                      idx_stride, num_tokens, num_heads, topk, sm_scale, out, max_logits, lse,
                                      stream);
}

}  // extern "C"

namespace dsa {

static int sparse_mla_prefill_impl(const void* q, int64_t q_token_stride, int64_t q_head_stride, const void* kv,
                                   int64_t kv_row_stride, int64_t s_kv, const int32_t* indices, int64_t idx_stride,
                                   int num_tokens, int num_heads, int topk, float sm_scale, void* out,
                                   float* max_logits, float* lse, void* stream) {
  if (num_tokens < 0 || num_heads <= 0 || (num_heads % 16) != 0)
    return set_error(kUnsupported, "sparse_mla_prefill: num_heads=%d must be a positive multiple of 16", num_heads);
  if (topk <= 0 || topk % 32 != 0)
    return set_error(kUnsupported, "sparse_mla_prefill: topk=%d must be a positive multiple of 32", topk);
  if (s_kv < 0 || s_kv > INT32_MAX)
    return set_error(kInvalidArgument, "sparse_mla_prefill: s_kv=%lld out of range", (long long)s_kv);
  if (num_tokens == 0) return kOk;
  if (!q || !indices || !out || (s_kv > 0 && !kv))
    return set_error(kInvalidArgument, "sparse_mla_prefill: null pointer");
  if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(kv) | reinterpret_cast<uintptr_t>(out)) & 15)
    return set_error(kInvalidArgument, "sparse_mla_prefill: q, kv and out must be 16-byte aligned");
  if ((q_token_stride % 8) || (q_head_stride % 8) || (kv_row_stride % 8) || kv_row_stride < 576)
    return set_error(kInvalidArgument, "sparse_mla_prefill: strides must be multiples of 8 elements, kv rows >= 576");
  return sparse_mla_rows_impl(q, q_token_stride, q_head_stride, kv, kv_row_stride, s_kv, indices, idx_stride,
                              num_tokens, num_heads, topk, sm_scale, out, max_logits, lse, stream);
}

static inline size_t pf_align(size_t x) { return (x + 255) & ~(size_t)255; }
static inline int cached_width(int topk) { return (topk + 63) / 64 * 64; }
static inline int fresh_width(int topk) { return (topk + 31) / 32 * 32; }

}  // namespace dsa

extern "C" {

size_t dsa_sparse_mla_prefill_paged_workspace_bytes(int num_tokens, int topk) {
  using namespace dsa;
  if (num_tokens <= 0 || topk <= 0) return 0;
  return pf_align((size_t)num_tokens * cached_width(topk) * 4) + pf_align((size_t)num_tokens * fresh_width(topk) * 4) +
         pf_align((size_t)num_tokens * 2 * 4);
}

int dsa_sparse_mla_prefill_paged(const void* q, int64_t q_token_stride, int64_t q_head_stride,
                                 const uint8_t* kv_cache, int64_t kv_block_stride_bytes, int kv_block_size,
                                 int64_t kv_num_blocks, const int32_t* block_table, int64_t bt_stride,
                                 int bt_width, const void* cu_seqlens_q, const void* cu_seqlens_k, int cu_is_64, int num_seqs,
                                 int64_t total_k, const void* fresh, int64_t fresh_row_stride, int64_t total_q,
                                 const int32_t* indices, int64_t idx_stride, int num_tokens, int num_heads, int topk,
                                 float sm_scale, void* out, float* max_logits, float* lse, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  using namespace dsa;
  if (num_tokens < 0 || num_seqs < 1 || total_k < 0 || total_q < 0 || topk <= 0 || kv_block_size <= 0 ||
      bt_width < 0 || bt_stride < bt_width)
    return set_error(kInvalidArgument, "sparse_mla_prefill_paged: bad sizes");
  if (num_tokens == 0) return kOk;
  if (!indices || !block_table || !cu_seqlens_q || !cu_seqlens_k || !out || !max_logits || !lse || !workspace)
    return set_error(kInvalidArgument, "sparse_mla_prefill_paged: null pointer");
  const size_t need = dsa_sparse_mla_prefill_paged_workspace_bytes(num_tokens, topk);
  if (workspace_bytes < need)
    return set_error(kWorkspaceTooSmall, "sparse_mla_prefill_paged: workspace %zu B < %zu B", workspace_bytes, need);
  const int cw = cached_width(topk), fw = fresh_width(topk);
  int32_t* cached = static_cast<int32_t*>(workspace);
  int32_t* fresh_idx =
      reinterpret_cast<int32_t*>(static_cast<uint8_t*>(workspace) + pf_align((size_t)num_tokens * cw * 4));
  int32_t* counts = reinterpret_cast<int32_t*>(static_cast<uint8_t*>(workspace) + pf_align((size_t)num_tokens * cw * 4) +
                                               pf_align((size_t)num_tokens * fw * 4));
  hipStream_t st = (hipStream_t)stream;
  // 1. each token's indices split into cache slots and fresh rows, compacted and counted
  hipLaunchKernelGGL(prefill_split_kernel, dim3((unsigned)num_tokens), dim3(256), 0, st, indices, idx_stride, topk,
                     cu_seqlens_q, cu_seqlens_k, cu_is_64, num_seqs, total_k, block_table, bt_stride, bt_width,
                     kv_block_size,
                     cached, cw, fresh_idx, fw, counts);
  if (int rc = check_launch("dsa_sparse_mla_prefill_paged(split)")) return rc;
  // 2. the decode kernel over each token's cache slots (fp8 rows, exact
  // dequantisation in registers) followed by its fresh bf16 rows, one softmax
  const MlaFresh fr{counts, fresh, fresh_row_stride, total_q, fresh_idx, fw};
  return sparse_mla_decode_impl(q, q_token_stride, q_head_stride, kv_cache, kv_block_stride_bytes, kv_block_size,
                                kv_num_blocks, cached, cw, num_tokens, num_heads, cw, sm_scale, out, lse, 1, nullptr, 0,
                                stream, max_logits, &fr);
}

}  // extern "C"
