// Page tables of sparse absorbed-MLA attention (DeepSeek sparse attention) on gfx950.
//
// An indexer hands over, per query token, the k cached tokens that it attends to.  The attention itself is the dense
// kernel of rpa_mla.hip over a page table of the token's own: these kernels write that table (one workgroup per query
// token) and put the token's new latent row where the dense kernel will find it, so that a call is three launches.
// (As tensor operations the same took 25 launches and 370 us of host time for 32 decode rows whose attention takes 40
// on the GPU; a token-level selection was also gathered, widened and copied once more: 5 x 75 MB for those rows.)
//
// What bounds them: latency.  A token's selection is 2 to 8 KB, read once; everything else happens in LDS.

#include "rpa_common.h"
#include "rpa_kernels.h"

namespace rpa {
namespace {

constexpr int kThreads = 256;
constexpr int kWords = 2048;  // bit map words in LDS: 65536 pages of a sequence at a time (4 M tokens in pages of 64)

// Sequence of query token `tok` (the last whose first token is <= tok; tokens past the end belong to the last one).
__device__ __forceinline__ int owner(const int32_t* cu_q_lens, int num_seqs, int tok) {
  int lo = 0, hi = num_seqs;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (scalar_load_i32(cu_q_lens + mid) <= tok) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Exclusive prefix sum of `x` over the workgroup; `total` = the sum.
__device__ __forceinline__ int block_scan(int x, int& total, int* wave_sums) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int incl = x;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int n = __shfl_up(incl, off);
    if (lane >= off) incl += n;
  }
  __syncthreads();  // the sums of an earlier scan have been read
  if (lane == 63) wave_sums[wave] = incl;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kThreads / 64; ++w) {
    if (w < wave) before += wave_sums[w];
    all += wave_sums[w];
  }
  total = all;
  return before + incl - x;
}

// One cached row of `a`'s layout from the new token's two parts (72 or 36 chunks of 16 bytes; the gap of a 640-wide
// row is left alone).
__device__ __forceinline__ void put_row(const SparseMlaArgs& a, char* row, int tok) {
  const int es = a.fp8 ? 1 : 2, t = threadIdx.x;
  if (t < 32 * es) st16(row + t * 16, ld16(a.new_kv_c + (int64_t)tok * 512 * es + t * 16));
  else if (t < 36 * es) st16(row + a.rope_offset * es + (t - 32 * es) * 16, ld16(a.new_k_pe + (int64_t)tok * 64 * es + (t - 32 * es) * 16));
}

// Whole pages: the distinct pages that a token's selection touches, ascending, at most k_pages_max - 1 of them and
// without the page of the new token, which comes last; the rest of the token's k_pages_max entries name the cache's
// last page.  The new row goes to its slot of the cache.
__global__ __launch_bounds__(kThreads) void rpa_sparse_pages_kernel(const SparseMlaArgs a) {
  __shared__ uint32_t bits[kWords];
  __shared__ int wave_sums[kThreads / 64];
  const int tok = blockIdx.x, tid = threadIdx.x;
  const int P = a.pt.page_size, kp = a.k_pages_max;
  const int seq = owner(a.pt.cu_q_lens, a.num_seqs, tok);
  const int kv_len = scalar_load_i32(a.pt.kv_lens + seq);
  const int page0 = scalar_load_i32(a.pt.cu_kv_lens + seq) / P;
  const int new_abs = max(kv_len - 1, 0), new_page = new_abs / P, new_off = new_abs - new_page * P;
  const int shift = (P & (P - 1)) == 0 ? 31 - __builtin_clz(P) : -1;
  auto physical = [&](int local) { return a.pt.page_indices[min(max(page0 + local, 0), a.num_page_indices - 1)]; };
  int32_t* out = a.table + (int64_t)tok * kp;
  const int32_t* sel = a.topk + (int64_t)tok * a.topk_stride;
  int hits = 0;
  for (int w0 = 0; w0 * 32 < a.pages_per_seq && hits < kp - 1; w0 += kWords) {
    const int words = min(kWords, (a.pages_per_seq + 31) / 32 - w0);
    for (int w = tid; w < words; w += kThreads) bits[w] = 0;
    __syncthreads();
    for (int j = tid; j < a.topk_count; j += kThreads) {
      const int idx = sel[j];
      const int page = a.topk_is_pages ? idx : (shift >= 0 ? idx >> shift : idx / P);
      const int bit = page - w0 * 32;
      if (idx >= 0 && page != new_page && page < a.pages_per_seq && bit >= 0 && bit < kWords * 32)
        atomicOr(&bits[bit >> 5], 1u << (bit & 31));
    }
    __syncthreads();
    for (int b0 = 0; b0 < words; b0 += kThreads) {
      uint32_t m = b0 + tid < words ? bits[b0 + tid] : 0u;
      int total;
      int at = hits + block_scan(__builtin_popcount(m), total, wave_sums);
      for (; m != 0 && at < kp - 1; m &= m - 1, ++at)
        out[at] = kv_len > 0 ? physical((w0 + b0 + tid) * 32 + __builtin_ctz(m)) : a.total_pages - 1;
      hits += total;
    }
    __syncthreads();
  }
  hits = min(hits, kp - 1);
  const int own = kv_len > 0 ? physical(new_page) : a.total_pages - 1;
  for (int j = hits + tid; j < kp; j += kThreads) out[j] = j == hits ? own : a.total_pages - 1;
  if (tid == 0) {
    a.kv_len_out[tok] = hits * P + new_off + 1;
    a.cu_q_out[tok] = tok;
    if (tok == a.num_tokens - 1) a.cu_q_out[tok + 1] = tok + 1;
  }
  if (a.new_kv_c) put_row(a, a.cache + ((int64_t)own * P + new_off) * a.row_stride * (a.fp8 ? 1 : 2), tok);
}

// Single tokens: the token's table names the rows of its selection (pages of one token, in the selection's order).
// The last valid entry is the new token itself, which the cache need not hold yet: its row is packed into `extra` and
// named there (page -1 - tok); an unused entry between valid ones names the row of zeros behind them.
__global__ __launch_bounds__(kThreads) void rpa_sparse_rows_kernel(const SparseMlaArgs a) {
  __shared__ int wave_sums[kThreads / 64];
  const int tok = blockIdx.x, tid = threadIdx.x;
  const int P = a.pt.page_size;
  const int seq = owner(a.pt.cu_q_lens, a.num_seqs, tok);
  const int page0 = scalar_load_i32(a.pt.cu_kv_lens + seq) / P;
  const int shift = (P & (P - 1)) == 0 ? 31 - __builtin_clz(P) : -1;
  const int32_t* sel = a.topk + (int64_t)tok * a.topk_stride;
  int32_t* out = a.table + (int64_t)tok * a.topk_count;
  int n = 0;
  for (int j0 = 0; j0 < a.topk_count; j0 += kThreads) {
    const int j = j0 + tid;
    const int idx = j < a.topk_count ? sel[j] : -1;
    if (j < a.topk_count) {
      const int local = shift >= 0 ? idx >> shift : idx / P;
      out[j] = idx < 0 ? -1 - a.num_tokens
                       : a.pt.page_indices[min(max(page0 + local, 0), a.num_page_indices - 1)] * P + (idx - local * P);
    }
    n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(idx >= 0));  // this wave's count
  }
  int total;
  block_scan((tid & 63) == 0 ? n : 0, total, wave_sums);  // (its barriers also order the table's writes below)
  const int es = a.fp8 ? 1 : 2;
  const int64_t row_bytes = (int64_t)a.row_stride * es;
  if (tid == 0) {
    if (a.new_kv_c && total > 0) out[total - 1] = -1 - tok;
    a.kv_len_out[tok] = total;
    a.cu_q_out[tok] = tok;
    if (tok == a.num_tokens - 1) a.cu_q_out[tok + 1] = tok + 1;
  }
  if (a.new_kv_c) put_row(a, a.extra + tok * row_bytes, tok);
  if (tok == 0)
    for (int64_t b = tid * 16; b < row_bytes; b += kThreads * 16) st16(a.extra + a.num_tokens * row_bytes + b, u32x4_t{0u, 0u, 0u, 0u});
}

}  // namespace

hipError_t launch_sparse_table(const SparseMlaArgs& a, hipStream_t stream) {
  if (a.num_tokens <= 0) return hipSuccess;
  if (a.k_pages_max > 0) hipLaunchKernelGGL(rpa_sparse_pages_kernel, dim3(a.num_tokens), dim3(kThreads), 0, stream, a);
  else hipLaunchKernelGGL(rpa_sparse_rows_kernel, dim3(a.num_tokens), dim3(kThreads), 0, stream, a);
  return hipGetLastError();
}

}  // namespace rpa
