// Page tables of sparse absorbed-MLA attention (DeepSeek sparse attention) on gfx950.
//
// An indexer hands over, per query token, the k cached tokens that it attends to.  The attention itself is the dense
// decode kernel of rpa_mla.hip over a page table of the token's own.  Each of its workgroups writes that table in front of its first
// copy, all of it and the same bytes as the other workgroups of the token (a row of the table starts a cache line of its own, so no
// line of it is in a cache before it is whole), and the workgroup that has the token's last tile puts the new latent row where it will
// find it.
//
// What bounds it: round trips to memory, one after the other.  A selection is 2 to 8 KB; it is requested in front of
// everything, beside the lengths and the search for the token's sequence, which are one load for up to 64 sequences, and the sequence's
// page ids arrive in LDS while the selection is sorted into its bit map.  Shared tiles take their page ids from there; the others read
// the table back.  As a launch in front of the attention's (what was here before) the tables took 7.2 us of the GPU, 4.3 for single
// rows, and 2.7 of the host.  The call, replayed from a graph / launched: 32 decode rows of 2048 entries x 16 heads, pages of 64
// 40.0 -> 36.7 / 44.3 -> 41.0 us, 4 rows of 1024 x 32 heads 25.1 -> 22.6, 20 rows x 128 heads on pages of 16 43.7 -> 41.2; single rows,
// 37 rows of 512 x 32 heads 24.1 -> 22.3, 22 of 2048 x 128 heads 49.1 -> 47.9.  With every kernel reading its ids from the table: 37.6..38.7
// for the first.
#pragma once

#include "rpa_common.h"
#include "rpa_kernels.h"

namespace rpa {
namespace sparse {

constexpr int kWords = 2048;  // bit map words in LDS: 65536 pages of a sequence at a time (4 M tokens in pages of 64)
constexpr int kList = 2048;   // pages of a table whose ids are looked up together (k_pages_max may be more)
constexpr int kBatch = 2048;  // entries of a selection that a workgroup requests at a time
constexpr int kSmall = 2048;  // pages of a sequence up to which its page ids wait in LDS, and a bit map is a word per lane

// A query token's row as the dense kernel sees it: its length, and where its new latent row belongs.
struct Row {
  int kv_len;
  char* fresh;
};

// A piece of a row: tokens [t_begin, t_end) of kv_len, those below t_lo behind the window.
struct Piece {
  int kv_len, t_lo, t_begin, t_end;
  int page_ids;  // lane's: of page t_begin / page size + lane, where the kernel keeps them in a register
};
__device__ __forceinline__ void cut(Piece& p, const MlaDecodeArgs& a, int split) {
  p.t_lo = a.sm.window > 0 ? max(0, p.kv_len - a.sm.window) : 0;
  p.t_begin = (p.t_lo & ~31) + split * a.chunk;  // (as the ordinary rows' pieces, and as the merge counts them)
  p.t_end = split == a.max_splits - 1 ? p.kv_len : min(p.kv_len, p.t_begin + a.chunk);
}

// What is known of the token's sequence (the last whose first token is <= tok; tokens past the end belong to the last one).
struct Owner {
  int kv_len, cu_kv;
};
__device__ __forceinline__ Owner owner(const SparseMlaArgs& a, int tok) {
  const int lane = threadIdx.x & 63, last = a.num_seqs - 1;
  Owner o;
  if (last < 64) {  // a sequence per lane
    const int s = min(lane, last);
    const int first = a.pt.cu_q_lens[s], kv = a.pt.kv_lens[s], cu = a.pt.cu_kv_lens[s];
    const int seq = __builtin_popcountll(__builtin_amdgcn_ballot_w64(lane >= 1 && lane <= last && first <= tok));
    o.kv_len = __builtin_amdgcn_readlane(kv, seq);
    o.cu_kv = __builtin_amdgcn_readlane(cu, seq);
    return o;
  }
  // cu_q_lens does not fall, so the first 64 whose last one starts behind the token decide
  int seq = 0;
  for (int s0 = 1; s0 <= last; s0 += 64) {
    const int s = s0 + lane;
    const int first = a.pt.cu_q_lens[min(s, last)];
    const int n = __builtin_popcountll(__builtin_amdgcn_ballot_w64(s <= last && first <= tok));
    seq += n;
    if (n < 64) break;
  }
  seq = __builtin_amdgcn_readfirstlane(seq);
  o.kv_len = scalar_load_i32(a.pt.kv_lens + seq);
  o.cu_kv = scalar_load_i32(a.pt.cu_kv_lens + seq);
  return o;
}

// Entries j0 + THREADS i + thread of a selection (-1 past its end).
template <int THREADS>
__device__ __forceinline__ void load_batch(int (&idx)[kBatch / THREADS], const int32_t* sel, int count, int j0) {
#pragma unroll
  for (int i = 0; i < kBatch / THREADS; ++i) {
    const int j = j0 + i * THREADS + (int)threadIdx.x;
    const int x = sel[min(j, count - 1)];
    idx[i] = j < count ? x : -1;
  }
}

// Exclusive prefix sum of `x` over the workgroup; `total` = the sum.
template <int THREADS>
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
  for (int w = 0; w < THREADS / 64; ++w) {
    if (w < wave) before += wave_sums[w];
    all += wave_sums[w];
  }
  total = __builtin_amdgcn_readfirstlane(all);  // (out of LDS: the compiler would take it, and every length and address after it, for the lane's own)
  return before + incl - x;
}

// Whole pages: the distinct pages that a token's selection touches, ascending, at most k_pages_max - 1 of them and
// without the page of the new token, which comes last; the rest of the token's k_pages_max entries name the cache's
// last page.  The new row belongs to its slot of the cache.
// IDS: the kernel keeps 64 page ids in a register (p.page_ids).  A piece of no more than that has no use for a table, and none is written.
template <int THREADS, bool IDS>
__device__ __forceinline__ Row pages_row(const MlaDecodeArgs& d, int tok, int split, char* lds, Piece& p) {
  const SparseMlaArgs& a = d.sparse;
  uint32_t* bits = reinterpret_cast<uint32_t*>(lds);
  int32_t* list = reinterpret_cast<int32_t*>(bits + kWords);  // the pages found, by their place in the sequence
  int32_t* phys = list + kList;                               // kSmall: the sequence's page ids
  int* wave_sums = list + kList;
  const int tid = threadIdx.x, lane = tid & 63;
  const int P = a.pt.page_size, kp = a.k_pages_max;
  const int32_t* sel = a.topk + (int64_t)tok * a.topk_stride;
  const bool small = a.pages_per_seq <= kSmall;
  int idx[kBatch / THREADS];
  if (a.topk_count > 0) load_batch<THREADS>(idx, sel, a.topk_count, 0);
  const Owner o = owner(a, tok);
  const int kv_len = o.kv_len, page0 = o.cu_kv / P;
  const int new_abs = max(kv_len - 1, 0), new_page = new_abs / P, new_off = new_abs - new_page * P;
  const int shift = (P & (P - 1)) == 0 ? 31 - __builtin_clz(P) : -1;
  auto physical = [&](int local) { return a.pt.page_indices[min(max(page0 + local, 0), a.num_page_indices - 1)]; };
  int id[kSmall / THREADS];
  if (small) {  // on their way while the selection is sorted
#pragma unroll
    for (int i = 0; i < kSmall / THREADS; ++i)
      if (i * THREADS < a.pages_per_seq) id[i] = physical(min(i * THREADS + tid, a.pages_per_seq - 1));
  }
  const int own = kv_len > 0 ? physical(new_page) : a.total_pages - 1;
  int32_t* out = a.table + (int64_t)tok * a.table_stride;
  auto mark = [&](int first, int limit) __attribute__((always_inline)) {  // the selection's pages first .. first + limit - 1
    for (int j0 = 0; j0 < a.topk_count; j0 += kBatch) {
      if (j0 > 0 || first > 0) load_batch<THREADS>(idx, sel, a.topk_count, j0);  // (the first batch is here already)
#pragma unroll
      for (int i = 0; i < kBatch / THREADS; ++i) {
        const int page = a.topk_is_pages ? idx[i] : (shift >= 0 ? idx[i] >> shift : idx[i] / P);
        const int bit = page - first;
        if (idx[i] >= 0 && page != new_page && page < a.pages_per_seq && bit >= 0 && bit < limit)
          atomicOr(&bits[bit >> 5], 1u << (bit & 31));
      }
    }
  };
  Row r;
  r.fresh = a.cache + ((int64_t)own * P + new_off) * a.row_stride * (a.fp8 ? 1 : 2);
  if (small) {
    if (tid < kSmall / 32) bits[tid] = 0;
    __syncthreads();
    mark(0, kSmall);
#pragma unroll
    for (int i = 0; i < kSmall / THREADS; ++i)
      if (i * THREADS < a.pages_per_seq) phys[i * THREADS + tid] = id[i];
    __syncthreads();
    // (every wave all of it, the same words: no barrier behind it)
    uint32_t m = bits[lane];
    const int found = __builtin_popcount(m);
    int incl = found;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int n = __shfl_up(incl, off);
      if (lane >= off) incl += n;
    }
    for (int at = incl - found; m != 0 && at < kp - 1 && at < kList; m &= m - 1, ++at) list[at] = lane * 32 + __builtin_ctz(m);
    asm volatile("" ::: "memory");
    const int hits = min(__builtin_amdgcn_readlane(incl, 63), kp - 1);
    auto id_at = [&](int j) { return kv_len > 0 ? j < hits ? phys[list[j]] : j == hits ? own : a.total_pages - 1 : a.total_pages - 1; };
    p.kv_len = r.kv_len = hits * P + new_off + 1;
    cut(p, d, split);
    const int first = p.t_begin / P;
    if constexpr (IDS) p.page_ids = id_at(min(first + lane, hits));
    // (copies are asked for up to five tiles ahead)
    if (!IDS || min(p.t_end + 160, p.kv_len) / P - first >= 64)
      for (int j = tid; j < kp; j += THREADS) out[j] = id_at(j);
    return r;
  }
  int hits = 0;
  for (int w0 = 0; w0 * 32 < a.pages_per_seq && hits < kp - 1; w0 += kWords) {
    const int words = min(kWords, (a.pages_per_seq + 31) / 32 - w0);
    for (int w = tid; w < words; w += THREADS) bits[w] = 0;
    __syncthreads();
    mark(w0 * 32, kWords * 32);
    __syncthreads();
    for (int b0 = 0; b0 < words; b0 += THREADS) {
      uint32_t m = b0 + tid < words ? bits[b0 + tid] : 0u;
      int total;
      int at = hits + block_scan<THREADS>(__builtin_popcount(m), total, wave_sums);
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
  for (int j = tid; j < min(hits, kList); j += THREADS) out[j] = kv_len > 0 ? physical(list[j]) : a.total_pages - 1;
  for (int j = hits + tid; j < kp; j += THREADS) out[j] = j == hits ? own : a.total_pages - 1;
  p.kv_len = r.kv_len = hits * P + new_off + 1;
  cut(p, d, split);
  if constexpr (IDS) {
    wait_all_loads();  // (and stores)
    __syncthreads();
    p.page_ids = out[min(p.t_begin / P + lane, hits)];
  }
  return r;
}

// Single tokens: the token's table names the rows of its selection (pages of one token, in the selection's order).
// The last valid entry is the new token itself, which the cache need not hold yet: its row belongs to `extra` and is
// named there (page -1 - tok); an unused entry between valid ones names the row of zeros behind them.
template <int THREADS>
__device__ __forceinline__ Row tokens_row(const SparseMlaArgs& a, int tok, char* lds) {
  int* wave_sums = reinterpret_cast<int*>(lds);
  const int tid = threadIdx.x;
  const int P = a.pt.page_size;
  const int32_t* sel = a.topk + (int64_t)tok * a.topk_stride;
  int idx[kBatch / THREADS];
  load_batch<THREADS>(idx, sel, a.topk_count, 0);
  const int page0 = owner(a, tok).cu_kv / P;
  const int shift = (P & (P - 1)) == 0 ? 31 - __builtin_clz(P) : -1;
  int32_t* out = a.table + (int64_t)tok * a.table_stride;
  // How many entries are valid comes first: the last of them is written as what it is, and once (the token's other workgroups write
  // the same bytes while this one may be reading already).
  int n = 0;
  for (int j0 = 0; j0 < a.topk_count; j0 += kBatch) {
    if (j0 > 0) load_batch<THREADS>(idx, sel, a.topk_count, j0);
#pragma unroll
    for (int i = 0; i < kBatch / THREADS; ++i) n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(idx[i] >= 0));  // this wave's count
  }
  int total;
  block_scan<THREADS>((tid & 63) == 0 ? n : 0, total, wave_sums);
  const int newest = a.new_kv_c ? total - 1 : -1;
  for (int j0 = 0; j0 < a.topk_count; j0 += kBatch) {
    if (a.topk_count > kBatch) load_batch<THREADS>(idx, sel, a.topk_count, j0);
    int row[kBatch / THREADS];
#pragma unroll
    for (int i = 0; i < kBatch / THREADS; ++i) {
      const int local = shift >= 0 ? idx[i] >> shift : idx[i] / P;
      row[i] = a.pt.page_indices[min(max(page0 + local, 0), a.num_page_indices - 1)] * P + (idx[i] - local * P);
    }
#pragma unroll
    for (int i = 0; i < kBatch / THREADS; ++i) {
      const int j = j0 + i * THREADS + tid;
      if (j < a.topk_count) out[j] = j == newest ? -1 - tok : idx[i] < 0 ? -1 - a.num_tokens : row[i];
    }
  }
  const int64_t row_bytes = (int64_t)a.row_stride * (a.fp8 ? 1 : 2);
  for (int64_t b = tid * 16; b < row_bytes; b += THREADS * 16) st16(a.extra + a.num_tokens * row_bytes + b, u32x4_t{0u, 0u, 0u, 0u});
  Row r;
  r.kv_len = total;
  r.fresh = a.extra + tok * row_bytes;
  return r;
}

// The new token's two parts as one cached row (72 or 36 chunks of 16 bytes; the gap of a 640-wide row is left alone): this thread's chunk,
// and where it goes.
__device__ __forceinline__ u32x4_t new_chunk(const SparseMlaArgs& a, int tok) {
  const int es = a.fp8 ? 1 : 2, t = min((int)threadIdx.x, 36 * es - 1);
  return ld16(t < 32 * es ? a.new_kv_c + (int64_t)tok * 512 * es + t * 16 : a.new_k_pe + (int64_t)tok * 64 * es + (t - 32 * es) * 16);
}
__device__ __forceinline__ void put_chunk(const SparseMlaArgs& a, char* row, u32x4_t x) {
  const int es = a.fp8 ? 1 : 2, t = threadIdx.x;
  if (t < 36 * es) st16(t < 32 * es ? row + t * 16 : row + a.rope_offset * es + (t - 32 * es) * 16, x);
}

// One piece of a query token's row on the fixed plan: what the piece takes, the table, and the new row if the row's last tile is in the
// piece.  false: nothing there.  The whole workgroup calls it; lds (24 KiB) is free again behind it.
template <int THREADS, bool IDS = false>
__device__ __forceinline__ bool begin_piece(const MlaDecodeArgs& a, int tok, int split, char* lds, Piece& p) {
  const SparseMlaArgs& s = a.sparse;
  u32x4_t fresh = {0u, 0u, 0u, 0u};
  if (s.new_kv_c) fresh = new_chunk(s, tok);
  Row r;
  if (s.k_pages_max > 0) {
    r = pages_row<THREADS, IDS>(a, tok, split, lds, p);
  } else {
    r = tokens_row<THREADS>(s, tok, lds);
    p.kv_len = r.kv_len;
    cut(p, a, split);
  }
  if (threadIdx.x == 0) s.kv_len_out[tok] = p.kv_len;  // (for the merge)
  if (p.t_begin >= p.kv_len) return false;
  if (s.new_kv_c && p.t_end == p.kv_len) put_chunk(s, r.fresh, fresh);
  wait_all_loads();  // (and stores)
  __syncthreads();
  return true;
}

}  // namespace sparse
}  // namespace rpa
