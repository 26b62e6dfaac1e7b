// Host-visible launch interface between the C ABI (rpa_capi.hip) and the
// kernel translation units.  Plain structs of device pointers and integers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rpa_shapes.h"
#include "rpa_tuning.h"

namespace rpa {

// How K and V rows of one (page, token, kv head) are addressed, in bytes.
//   fused  [pages, P, 2*Hkv, D]: v_base = k_base + D*esize, head_stride = 2*D*esize
//   split  k_pages / v_pages [pages, P, Hkv, D]: head_stride = D*esize
struct KvAddr {
  const char* k_base;
  const char* v_base;
  int64_t page_stride;
  int32_t tok_stride;
  int32_t head_stride;
};

struct PageTable {
  const int32_t* kv_lens;
  const int32_t* page_indices;
  const int32_t* cu_q_lens;
  const int32_t* cu_kv_lens;  // nullptr => padded table, row stride pages_per_seq
  int32_t pages_per_seq;
  int32_t page_size;
};

struct SoftmaxOpts {
  float sm_scale;
  float soft_cap;    // 0 => off
  float mask_value;  // finite, negative
  int32_t window;    // 0 => off
  const float* sink;  // f32[Hq] extra logit per query head that only enters the denominator, or nullptr
  float xai_len;      // > 0: logits of a query at position p > xai_len are multiplied by log2(p)/log2(xai_len)
  // prefill kernels only: 0 causal, 1 custom mask, 2 no mask
  int32_t mask_mode;
  int32_t mask_rows_page_aligned;
  const int32_t* custom_mask;
  const int32_t* cu_mask_lens;
  int32_t round_logits;  // masked logits and the sink are rounded before the softmax: 1 to bf16, 2 to f16
  float q_scale;         // > 0: queries are divided by it and rounded to the cache's element type; 0 => off
};

struct DecodeArgs {
  const uint16_t* q;  // bf16 [T, Hq, D]
  uint16_t* out;      // bf16 [T, Hq, D]
  KvAddr kv;
  PageTable pt;
  SoftmaxOpts sm;
  const float* k_scale;  // f32[Hkv] or nullptr
  const float* v_scale;
  float* ws_o;   // [num_rows, max_splits, Hq, D] unnormalised partial outputs
  float* ws_ml;  // [num_rows, max_splits, Hq, 2]  (running max in log2 units, sum)
  int32_t num_rows;  // decode sequences
  int32_t Hq, Hkv, G;
  int32_t q_dim;       // elements of a row of q, out, new_k, new_v (<= the head dim of the cache, whose rest is zero)
  int32_t chunk;       // fixed plan: kv tokens per split (multiple of 32)
  int32_t max_splits;  // fixed plan: grid.x
  int32_t fp8;
  // balanced plan: every wave takes the same number of 32-token blocks of the whole batch;
  // ws_o / ws_ml hold 2 * num_wgs * waves_per_wg groups of 16 rows
  int32_t balanced;
  int32_t num_wgs;       // workgroups of the balanced grid
  int32_t waves_per_wg;  // neighbouring kv heads walked together
  int32_t min_blocks_per_wave;
  int32_t forced_blocks_per_wave;  // > 0: tests pin the partition
  int32_t* cu_blocks;              // [num_rows + 1] prefix sum of 32-token blocks, written by the kernel
  // balanced plan, merge inside the kernel: one arrival word per (row, unit, wave of the
  // workgroup), [generation : 48 | arrivals : 16]; nullptr => a second launch merges
  unsigned long long* merge_counters;
  unsigned long long generation;  // of this call; a word of another generation counts as zero
  // device i32[3] (decode_end, prefill_end, num_seqs) or nullptr: when given, num_rows is only a bound
  // and the rows to process are [0, min(num_rows, dist[0]))
  const int32_t* dist;
  // New tokens that are not in the cache yet, [T, Hkv, D] in its element type, or nullptr: the kernel reads them from
  // here and leaves each in its cache slot
  const char* new_k;
  const char* new_v;
  int32_t token_rows;    // fixed plan: rows are the query tokens of sequences [0, num_seqs), of any length
  int32_t num_seqs;      // token_rows: sequences (with dist: a bound on dist[2])
  int32_t group_rows;    // fixed plan: one workgroup per (row, kv head, piece), merged in LDS (rpa_decode_row_kernel)
};

// New tokens on their way into the cache.
struct KvWriteArgs {
  KvAddr kv;  // bases are written through
  PageTable pt;
  const char* keys;    // [T, Hkv, D] cache dtype
  const char* values;
  int32_t num_seqs;
  int32_t Hkv;
  int32_t head_bytes;
  int32_t src_head_bytes;  // of a head in keys / values (<= head_bytes; the rest of the cached row is set to zero)
  int32_t num_tokens;
  const int32_t* dist;  // device i32[3] or nullptr: when given, num_seqs is only a bound on dist[2]
  // decode rows whose tokens the decode kernel writes itself are left out: sequences [0, seq_begin), with dist
  // (skip_decode_rows) sequences [0, dist[0])
  int32_t seq_begin;
  int32_t skip_decode_rows;
};

struct FastDiv {
  uint32_t mul, shift;
};

struct PrefillArgs {
  const uint16_t* q;
  uint16_t* out;
  KvAddr kv;
  PageTable pt;
  SoftmaxOpts sm;
  const float* k_scale;
  const float* v_scale;
  int32_t seq_begin, seq_end;  // sequences [seq_begin, seq_end)
  int32_t Hq, Hkv, G;
  int32_t q_dim;       // elements of a row of q and out (<= head_dim)
  int32_t max_q_len;
  int32_t max_kv_len;  // host bound on kv_len of these sequences, 0 = unknown
  int32_t fp8;
  int32_t head_dim;  // 128, or 256 (bf16 cache only)
  // device i32[3] or nullptr: when given, seq_end is only a bound and the sequences to process are
  // [dist[0], min(seq_end, dist[2])) (custom-mask calls: [0, ...))
  const int32_t* dist;
  // K/V range of every workgroup cut into kv_splits pieces (pipelined kernel, launches that would leave most
  // of the GPU idle; 0 or 1 = whole ranges): partial rows f32 [token][Hq][piece][128] in ws_o, their
  // (reference, sum) pairs in ws_ml, merged by a second launch over num_tokens x Hq rows
  int32_t kv_splits;
  int32_t num_tokens;  // bound on the query tokens of the call (rows of q)
  float* ws_o;
  float* ws_ml;
  // Custom masks: one bit per (query token, kv token), mask_pitch 64-bit words per token row, written by
  // rpa_mask_bits_kernel in front of the attention kernels (with write.keys it also puts the new tokens into the
  // cache); nullptr: the kernels read the caller's i32 words
  uint64_t* mask_bits;
  int32_t mask_pitch;
  // Prompts without a prefix: kv addresses the caller's new rows (a sequence's start at its first query token, one huge
  // page), and the last write_blocks workgroups of the grid put them into the cache, write_tokens each.
  int32_t rows_are_new;
  int32_t write_blocks, write_tokens;
  KvWriteArgs write;
  // ShapeOption bits of the cache's pages (for the launchers).  They choose the kernel also where it reads the caller's
  // rows, which would suit any: the assembly kernel rounds the scaled queries to bf16, and pages that it does not take
  // never had that
  uint32_t page_options;
  // The new tokens are not in the cache yet: rpa_prefill_packed_kernel reads those behind a sequence's prefix from write.keys /
  // write.values, and the last write_blocks workgroups put them into the cache.
  int32_t tail_is_new;
  int32_t mask_words;  // custom masks: rpa_prefill_packed_kernel reads the caller's words itself, no bits are made
  int32_t saves_launch;  // (for the choice) rpa_prefill_packed_kernel would spare the launch that writes the new tokens
  int32_t packed;  // rpa_prefill_packed_kernel takes the call, K/V ranges in so many pieces where there is room for them; 0 = not
  struct {
    FastDiv groups, units, hkv, per_kv, nseq;
    int32_t apart;
    int32_t block;  // > 0: so many tiles of a sequence one after the other (the order by streams)
    FastDiv round, seq_round, run;
  } map;  // set by the launchers (prefill_grid)
};

struct GatherArgs {
  KvAddr kv;
  PageTable pt;
  int32_t seq;
  int32_t row_bytes;  // Hkv * D * esize of one gathered K (or V) row
  int32_t Hkv;
  int32_t head_bytes;  // D * esize
  void* k_out;
  void* v_out;
  int32_t max_tokens;
};

// Sparse MLA: every query token is a decode row over a page table of its own, which the attention kernels write (rpa_dsa.h).
struct SparseMlaArgs {
  PageTable pt;              // of the batch: ragged table (cu_kv_lens)
  int32_t num_page_indices;  // entries of pt.page_indices
  int32_t num_tokens;
  int32_t num_seqs;
  const int32_t* topk;       // [T, topk_stride], the first topk_count of a row are read; -1 = unused
  int32_t topk_count, topk_stride;
  int32_t topk_is_pages;     // entries are pages of the sequence, not tokens
  int32_t pages_per_seq;
  int32_t k_pages_max;       // > 0: tables of whole pages; 0: tables of single rows
  int32_t total_pages;
  char* cache;               // whole pages: the new rows are written here
  int32_t row_stride, rope_offset, fp8;
  const char* new_kv_c;      // [T, 512] in the cache's element type, or nullptr: the cache holds them already
  const char* new_k_pe;      // [T, 64]
  int32_t* table;            // [T, table_stride], k_pages_max or topk_count entries of each row
  int32_t table_stride;      // a multiple of 32: no two rows share a cache line
  int32_t* kv_len_out;       // [T]
  char* extra;               // single rows: [T + 1] rows, the new ones and one of zeros
};

struct MlaDecodeArgs {
  const uint16_t* ql_nope;  // [T, Hq, lkv]
  const uint16_t* q_pe;     // [T, Hq, rope]
  uint16_t* out;            // [T, Hq, lkv]
  const char* cache;        // [pages, P, row_stride] bf16 or e4m3
  PageTable pt;
  SoftmaxOpts sm;
  uint16_t* ws_o;  // [T, max_splits, Hq, lkv] unnormalised partial outputs, bf16
  float* ws_ml;    // [T, max_splits, Hq, 2] (reference in log2 units, sum)
  int32_t num_rows;     // grid rows: sequences (rows_are_tokens == 0) or query tokens
  int32_t num_seqs;
  int32_t rows_are_tokens;  // 1: row r is query token r of whatever sequence owns it (any q_len)
  int32_t Hq;
  int32_t row_stride;   // elements
  int32_t rope_offset;  // elements
  int32_t chunk;
  int32_t max_splits;
  // balanced plan (sequence rows only): the workgroups share the 32-token tiles of the batch
  // evenly; ws_o / ws_ml hold 2 * num_wgs groups of 128 heads
  int32_t balanced;
  int32_t num_wgs;
  int32_t min_tiles_per_wg;
  int32_t forced_tiles_per_wg;
  int32_t waves;      // the kernels of a wave per tile (rpa_mla_waves.hip), 16 heads per workgroup
  int32_t siblings;   // workgroups that take the same share or piece, each for heads of its own (rpa_mla_waves.hip); 1 elsewhere
  int32_t piece_pad;  // balanced plan: what starting one more (row, head group) costs a workgroup, in tiles
  int32_t* cu_tiles;  // [num_rows + 1] prefix sum of tiles, written by the kernel
  float out_scale;    // finished rows are multiplied by it (v_scale; 1 when off)
  const int32_t* dist;  // device i32[3] or nullptr: when given, num_seqs is only a bound on dist[2]
  int32_t fp8;          // cache rows are e4m3 bytes (row_stride / rope_offset stay in elements)
  // pages -1, -2, ... of the page table are pages 0, 1, ... of this buffer (pages under 32 tokens only), or nullptr
  const char* extra_rows;
  // sequence rows: the new tokens' latents, [T, 512] and [T, 64] in the cache's type, which the kernels put into the cache; or nullptr
  const char* new_kv_c;
  const char* new_k_pe;
  SparseMlaArgs sparse;  // sparse.topk: the rows' page tables and lengths (pt) are still to be written, new rows are sparse.new_kv_c
};

struct MlaWriteArgs {
  char* cache;              // [pages, P, row_stride] bf16
  PageTable pt;
  const char* new_kv_c;  // [T, 512] in the cache's element type
  const char* new_k_pe;  // [T, 64]
  int32_t fp8;
  int32_t num_tokens;
  int32_t num_seqs;
  int32_t row_stride;
  int32_t rope_offset;
  const int32_t* dist;  // device i32[3] or nullptr: when given, num_seqs is only a bound on dist[2]
};

hipError_t launch_decode(const DecodeArgs& a, hipStream_t stream);
hipError_t launch_prefill(const PrefillArgs& a, hipStream_t stream);
// How many pieces launch_prefill would cut the K/V ranges into if it had the workspace (1 = no cut), and the
// bytes of workspace that takes.
int prefill_kv_splits(const PrefillArgs& a);
int prefill_packed_pieces(const PrefillArgs& a);
int compute_units();  // of the current device (256 where there is none)
size_t prefill_split_workspace_bytes(const PrefillArgs& a, int splits);
// n host words to device memory, in stream order; the source may be reused at once
hipError_t launch_upload(int32_t* dst, const int32_t* src, int n, hipStream_t stream);
hipError_t launch_gather(const GatherArgs& a, hipStream_t stream);
// head_dim 256: every query token of sequences [seq_begin, seq_end) as a row of its own; at most
// max_token_rows tokens (a host bound) are covered.  With a.dist set, seq_end is a bound and dist_role says
// which partition the kernel takes from the device: 1 = decode rows, 2 = everything behind them
hipError_t launch_rows256(const DecodeArgs& a, int seq_begin, int seq_end, int max_token_rows, int dist_role,
                          hipStream_t stream);
hipError_t launch_kv_write(const KvWriteArgs& a, hipStream_t stream);
hipError_t launch_mla_decode(const MlaDecodeArgs& a, hipStream_t stream);
hipError_t launch_mla_waves(const MlaDecodeArgs& a, hipStream_t stream);
// The rows of the shape table (rpa_shapes.h) these launchers select for a call, RPA_* overrides applied.
const ShapeRule& prefill_shape_of(const PrefillArgs& a);
// Whether launch_prefill would take long sequences one after the other (streams_in_turn, rpa_prefill_common.h).
bool prefill_by_streams(const PrefillArgs& a);
ShapeKey mla_shape_key(const MlaDecodeArgs& a);
unsigned mla_shape_skip(const MlaDecodeArgs& a, const Tuning& tune);
// how query tokens of a chunk share a workgroup (0: they do not; 1, 2: eight waves; 3: wide workgroups)
int mla_token_group_mode(const MlaDecodeArgs& a, const Tuning& tune, const ShapeRule& shape);
bool mla_takes_wide_p16(const MlaDecodeArgs& a, bool heads_in_128s);
hipError_t launch_mla_kv_write(const MlaWriteArgs& a, hipStream_t stream);

}  // namespace rpa
