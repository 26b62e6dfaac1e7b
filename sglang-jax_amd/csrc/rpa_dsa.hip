// Page tables of sparse absorbed-MLA attention (DeepSeek sparse attention) on gfx950.
//
// An indexer hands over, per query token, the k cached tokens that it attends to.  The attention itself is the dense
// kernel of rpa_mla.hip over a page table of the token's own: these kernels write that table (one workgroup per query
// token) and put the token's new latent row where the dense kernel will find it, so that a call is three launches.
// (As tensor operations the same took 25 launches and 370 us of host time for 32 decode rows whose attention takes 40
// on the GPU; a token-level selection was also gathered, widened and copied once more: 5 x 75 MB for those rows.)
//
// What bounds them: round trips to memory, one after the other.  A token's selection is 2 to 8 KB; it is requested in front of
// everything, kBatch entries per thread at a time, beside the search for the token's sequence, which is one load for up to 64
// sequences, and the pages it names are requested together.  Entry by entry behind a binary search (what was here before) the
// table of 32 decode rows, 2048 entries each, took 9.8 us; now 7.1 (what is left: the launch, three dependent round trips, LDS).

#include "rpa_common.h"
#include "rpa_kernels.h"

namespace rpa {
namespace {

constexpr int kThreads = 256;
constexpr int kWords = 2048;  // bit map words in LDS: 65536 pages of a sequence at a time (4 M tokens in pages of 64)

constexpr int kList = 2048;   // pages of a table whose ids are looked up together (k_pages_max may be more)
constexpr int kBatch = 8;     // entries of a selection that a thread requests at a time

// Sequence of query token `tok` (the last whose first token is <= tok; tokens past the end belong to the last one).
// A few by scalar loads; else 64 at a time: cu_q_lens does not fall, so the first 64 whose last one starts behind the token
// decide.
__device__ __forceinline__ int owner(const int32_t* cu_q_lens, int num_seqs, int tok) {
  if (num_seqs <= 4) {
    int n = 0;
    for (int s = 1; s < num_seqs; ++s) n += scalar_load_i32(cu_q_lens + s) <= tok ? 1 : 0;
    return n;
  }
  const int lane = threadIdx.x & 63;
  int seq = 0;
  for (int s0 = 1; s0 < num_seqs; s0 += 64) {
    const int s = s0 + lane;
    const int first = cu_q_lens[min(s, num_seqs - 1)];
    const int n = __builtin_popcountll(__builtin_amdgcn_ballot_w64(s < num_seqs && first <= tok));
    seq += n;
    if (n < 64) break;
  }
  return __builtin_amdgcn_readfirstlane(seq);
}

// Entries j0 + 256 i + thread of a selection, i = 0 .. kBatch - 1 (-1 past its end).
__device__ __forceinline__ void load_batch(int (&idx)[kBatch], const int32_t* sel, int count, int j0) {
#pragma unroll
  for (int i = 0; i < kBatch; ++i) {
    const int j = j0 + i * kThreads + (int)threadIdx.x;
    const int x = sel[min(j, count - 1)];
    idx[i] = j < count ? x : -1;
  }
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
// row is left alone): this thread's chunk, and where it goes.
__device__ __forceinline__ u32x4_t new_chunk(const SparseMlaArgs& a, int tok) {
  const int es = a.fp8 ? 1 : 2, t = min((int)threadIdx.x, 36 * es - 1);
  return ld16(t < 32 * es ? a.new_kv_c + (int64_t)tok * 512 * es + t * 16 : a.new_k_pe + (int64_t)tok * 64 * es + (t - 32 * es) * 16);
}
__device__ __forceinline__ void put_chunk(const SparseMlaArgs& a, char* row, u32x4_t x) {
  const int es = a.fp8 ? 1 : 2, t = threadIdx.x;
  if (t < 36 * es) st16(t < 32 * es ? row + t * 16 : row + a.rope_offset * es + (t - 32 * es) * 16, x);
}

// Whole pages: the distinct pages that a token's selection touches, ascending, at most k_pages_max - 1 of them and
// without the page of the new token, which comes last; the rest of the token's k_pages_max entries name the cache's
// last page.  The new row goes to its slot of the cache.
__global__ __launch_bounds__(kThreads) void rpa_sparse_pages_kernel(const SparseMlaArgs a) {
  __shared__ uint32_t bits[kWords];
  __shared__ int32_t list[kList];  // the pages found, by their place in the sequence
  __shared__ int wave_sums[kThreads / 64];
  const int tok = blockIdx.x, tid = threadIdx.x;
  const int P = a.pt.page_size, kp = a.k_pages_max;
  const int32_t* sel = a.topk + (int64_t)tok * a.topk_stride;
  int idx[kBatch];
  if (a.topk_count > 0) load_batch(idx, sel, a.topk_count, 0);
  u32x4_t fresh = {0u, 0u, 0u, 0u};
  if (a.new_kv_c) fresh = new_chunk(a, tok);
  const int seq = owner(a.pt.cu_q_lens, a.num_seqs, tok);
  const int kv_len = scalar_load_i32(a.pt.kv_lens + seq);
  const int page0 = scalar_load_i32(a.pt.cu_kv_lens + seq) / P;
  const int new_abs = max(kv_len - 1, 0), new_page = new_abs / P, new_off = new_abs - new_page * P;
  const int shift = (P & (P - 1)) == 0 ? 31 - __builtin_clz(P) : -1;
  auto physical = [&](int local) { return a.pt.page_indices[min(max(page0 + local, 0), a.num_page_indices - 1)]; };
  const int own = kv_len > 0 ? physical(new_page) : a.total_pages - 1;
  int32_t* out = a.table + (int64_t)tok * kp;
  int hits = 0;
  for (int w0 = 0; w0 * 32 < a.pages_per_seq && hits < kp - 1; w0 += kWords) {
    const int words = min(kWords, (a.pages_per_seq + 31) / 32 - w0);
    for (int w = tid; w < words; w += kThreads) bits[w] = 0;
    __syncthreads();
    for (int j0 = 0; j0 < a.topk_count; j0 += kBatch * kThreads) {
      if (j0 > 0 || w0 > 0) load_batch(idx, sel, a.topk_count, j0);  // (the first batch is here already)
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const int page = a.topk_is_pages ? idx[i] : (shift >= 0 ? idx[i] >> shift : idx[i] / P);
        const int bit = page - w0 * 32;
        if (idx[i] >= 0 && page != new_page && page < a.pages_per_seq && bit >= 0 && bit < kWords * 32)
          atomicOr(&bits[bit >> 5], 1u << (bit & 31));
      }
    }
    __syncthreads();
    for (int b0 = 0; b0 < words; b0 += kThreads) {
      uint32_t m = b0 + tid < words ? bits[b0 + tid] : 0u;
      int total;
      int at = hits + block_scan(__builtin_popcount(m), total, wave_sums);
      for (; m != 0 && at < kp - 1; m &= m - 1, ++at) {
        const int page = (w0 + b0 + tid) * 32 + __builtin_ctz(m);
        if (at < kList) list[at] = page;
        else out[at] = kv_len > 0 ? physical(page) : a.total_pages - 1;
      }
      hits += total;
    }
    __syncthreads();
  }
  hits = min(hits, kp - 1);
  // (behind the loop's last barrier.  A word's pages are neighbours: looked up where they are found, by one thread, they
  // were a chain of up to 32 round trips)
  for (int j = tid; j < min(hits, kList); j += kThreads) out[j] = kv_len > 0 ? physical(list[j]) : a.total_pages - 1;
  for (int j = hits + tid; j < kp; j += kThreads) out[j] = j == hits ? own : a.total_pages - 1;
  if (tid == 0) {
    a.kv_len_out[tok] = hits * P + new_off + 1;
    a.cu_q_out[tok] = tok;
    if (tok == a.num_tokens - 1) a.cu_q_out[tok + 1] = tok + 1;
  }
  if (a.new_kv_c) put_chunk(a, a.cache + ((int64_t)own * P + new_off) * a.row_stride * (a.fp8 ? 1 : 2), fresh);
}

// Single tokens: the token's table names the rows of its selection (pages of one token, in the selection's order).
// The last valid entry is the new token itself, which the cache need not hold yet: its row is packed into `extra` and
// named there (page -1 - tok); an unused entry between valid ones names the row of zeros behind them.
__global__ __launch_bounds__(kThreads) void rpa_sparse_rows_kernel(const SparseMlaArgs a) {
  __shared__ int wave_sums[kThreads / 64];
  const int tok = blockIdx.x, tid = threadIdx.x;
  const int P = a.pt.page_size;
  const int32_t* sel = a.topk + (int64_t)tok * a.topk_stride;
  int idx[kBatch];
  load_batch(idx, sel, a.topk_count, 0);
  u32x4_t fresh = {0u, 0u, 0u, 0u};
  if (a.new_kv_c) fresh = new_chunk(a, tok);
  const int seq = owner(a.pt.cu_q_lens, a.num_seqs, tok);
  const int page0 = scalar_load_i32(a.pt.cu_kv_lens + seq) / P;
  const int shift = (P & (P - 1)) == 0 ? 31 - __builtin_clz(P) : -1;
  int32_t* out = a.table + (int64_t)tok * a.topk_count;
  int n = 0;
  for (int j0 = 0; j0 < a.topk_count; j0 += kBatch * kThreads) {
    if (j0 > 0) load_batch(idx, sel, a.topk_count, j0);
    int row[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int local = shift >= 0 ? idx[i] >> shift : idx[i] / P;
      row[i] = a.pt.page_indices[min(max(page0 + local, 0), a.num_page_indices - 1)] * P + (idx[i] - local * P);
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int j = j0 + i * kThreads + tid;
      if (j < a.topk_count) out[j] = idx[i] < 0 ? -1 - a.num_tokens : row[i];
      n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(idx[i] >= 0));  // this wave's count
    }
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
  if (a.new_kv_c) put_chunk(a, a.extra + tok * row_bytes, fresh);
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
