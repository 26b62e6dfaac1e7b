// What the kernels of absorbed MLA share (rpa_mla.hip, rpa_mla_waves.hip): what a grid row attends to, where its result goes, how a ragged
// batch is dealt out to the workgroups.
#pragma once

#include "rpa_common.h"
#include "rpa_kernels.h"

namespace rpa {

// Per-workgroup timestamps of the wide balanced kernel, compiled in with -DRPA_MLA_TRACE only (build.py passes
// extra flags through): for up to four pieces per workgroup the 100 MHz clock at piece entry, first tiles and
// queries landed, tile loop entered, tile loop left, rows written.  rpa_debug_mla_trace() copies them out.
#ifdef RPA_MLA_TRACE
static __device__ unsigned long long rpa_mla_trace_buf[1024][4][8];
#define RPA_MLA_STAMP(slot)                                                                              \
  do {                                                                                                   \
    if (threadIdx.x == 0 && trace_piece < 4) rpa_mla_trace_buf[blockIdx.x & 1023][trace_piece][slot] = wall_clock64(); \
  } while (0)
#else
#define RPA_MLA_STAMP(slot) do { } while (0)
#endif

namespace {

constexpr int kTok = 32;                 // tokens per tile

__device__ __forceinline__ u32x4_t lds_ld16(const char* p) { return *reinterpret_cast<const u32x4_t*>(p); }

typedef uint32_t u32x32_t __attribute__((ext_vector_type(32)));
typedef uint32_t u32x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x32_t __attribute__((ext_vector_type(32)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2_t lds_tr16(const char* p) {
  typedef __attribute__((address_space(3))) s16x4_t* lds_ptr_t;
  const s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)(p));
  return __builtin_bit_cast(u32x2_t, v);
}

// The lane id behind a fence the compiler cannot see through: values derived from it are not common
// subexpressions of anything earlier, so they are worked out again where they are used instead of being
// kept in registers across code that has none to spare (the assembly loop pins 251 of a wave's 256; with
// them carried over it, 23-37 registers went to scratch memory per segment, 100 MB a launch on a
// prefill batch).  Counted by two instructions of its own, not taken from threadIdx, which would itself be kept in scratch memory across
// the loops.
__device__ __forceinline__ int fresh_lane() {
  int ln;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
  return ln;
}

// token (inside a tile) behind slot i = 4b + r of lane group g in the S^T result registers
__device__ __forceinline__ int tok_of(int g, int i) {
  return 16 * (i >> 2) + 4 * g + (i & 3);
}

// Sequence that owns query token `row`: the last one whose first token is <= row
// (zero-length sequences are skipped).  cu_q_lens[0 .. num_seqs] is non-decreasing.
__device__ __forceinline__ int owner_of_token(const int32_t* cu_q_lens, int num_seqs, int row) {
  int lo = 0, hi = num_seqs;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (scalar_load_i32(cu_q_lens + mid) <= row) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Query tokens are taken last first: a chunk's last tokens see the most, and what starts last should be short.  1405 tokens x
// 64 heads e4m3 124 -> 101 us, 6 prompts of 88 .. 307 tokens x 128 heads 137 -> 127, 900 tokens x 128 heads 164 -> 158.
//
// What a grid row attends to.  Sequence rows (decode batches): the one query of sequence `row`
// sees all kv_len tokens.  Token rows: query token `row` of a sequence with q_len new tokens
// sits at position kv_len - q_len + j and sees the tokens up to itself -- an absorbed-MLA
// prefill row is a decode row over a shorter prefix (mla/v1/ref.py:229-233).
struct MlaRow {
  int seq, kv_len, tq;
  bool valid;
};

__device__ __forceinline__ MlaRow mla_row(const MlaDecodeArgs& a, int row) {
  MlaRow r;
  r.valid = true;
  // static-shape mode: num_seqs is a bound, the number of sequences comes from the device
  const int num_seqs = a.dist ? min(a.num_seqs, scalar_load_i32(a.dist + 2)) : a.num_seqs;
  if (a.rows_are_tokens) {
    if (row >= scalar_load_i32(a.pt.cu_q_lens + num_seqs)) {
      r.valid = false;
      r.seq = r.kv_len = r.tq = 0;
      return r;
    }
    r.seq = owner_of_token(a.pt.cu_q_lens, num_seqs, row);
    const int q0 = scalar_load_i32(a.pt.cu_q_lens + r.seq);
    const int q_len = scalar_load_i32(a.pt.cu_q_lens + r.seq + 1) - q0;
    r.kv_len = scalar_load_i32(a.pt.kv_lens + r.seq) - q_len + (row - q0) + 1;
    r.tq = row;
  } else {
    r.seq = row;
    r.kv_len = (row < num_seqs) ? a.pt.kv_lens[row] : 0;
    r.tq = a.sparse.topk ? row : a.pt.cu_q_lens[row];
    r.valid = row < num_seqs;
  }
  return r;
}

// Where a workgroup leaves the result of one piece of work: finished bf16 rows in `out`, or
// unnormalised partial rows plus (max, sum) in workspace slot `base` + head.
struct MlaDest {
  bool final_rows;
  int64_t base;
};

// A sequence row's new token, from the caller's rows into the cache (a.new_kv_c), by every workgroup whose share holds the row's last
// tile, in front of everything else that it does.  A launch of its own for 1152 bytes a row took 5.4 us of the GPU and 2.7 of the
// host; here it is a round trip to memory at the start of those workgroups: 64 ragged rows x 128 heads 179.8 -> 177.4 us, 25 rows of
// 125..1062 38.0 -> 35.8, 2 of 4516..9525 x 16 heads 32.3 -> 30.2, 6 of 351..927 e4m3 33.7 -> 30.7.  Many short rows, each of which
// pays that round trip, are no slower: 600 rows of 100..200 x 128 heads 95.5 -> 94.2, 1000 of 30..100 118.6 -> 117.8, e4m3 121.4 -> 116.0.
// Every wave writes the whole row (the same bytes, 2 stores), so the copies that it makes of it afterwards follow its own stores
// and no barrier is needed.  Tiles behind a piece's first three are asked for behind a wait for the first one, which is younger than
// the stores; where the row's last tile may be among the first three the caller of this waits for the stores.  (Registers that
// wait for the token beside the first copies are live into the tile loops, which spill then and drain their copies to
// reload: 22 rows on token-level selections x 128 heads, which bring no token here, 50.3 -> 52.3 us.)
template <bool FP8>
__device__ __forceinline__ void put_new_row(const MlaDecodeArgs& a, int seq, int kv_len) {
  const int lane = threadIdx.x & 63;
  const int P = a.pt.page_size;
  const int q0 = scalar_load_i32(a.pt.cu_q_lens + seq), n = scalar_load_i32(a.pt.cu_q_lens + seq + 1) - q0;
  const int32_t* pages = a.pt.page_indices + (a.pt.cu_kv_lens ? (int64_t)(scalar_load_i32(a.pt.cu_kv_lens + seq) / P)
                                                            : (int64_t)seq * a.pt.pages_per_seq);
  for (int j = 0; j < n; ++j) {  // (one: a decode row brings one token)
    const int64_t tok = q0 + j;
    const int pos = kv_len - n + j;
    if (pos < 0) continue;
    const int slot = __builtin_amdgcn_readfirstlane((P & (P - 1)) == 0 ? pos >> (31 - __builtin_clz(P)) : pos / P);
    char* page = const_cast<char*>(a.cache);
    if constexpr (FP8) {
      const int t = min(lane, 35);
      const u32x4_t x = ld16(t < 32 ? a.new_kv_c + tok * 512 + t * 16 : a.new_k_pe + tok * 64 + (t - 32) * 16);
      char* row = page + ((int64_t)scalar_load_i32(pages + slot) * P + (pos - slot * P)) * a.row_stride;
      if (lane < 36) st16(row + (lane < 32 ? lane * 16 : a.rope_offset + (lane - 32) * 16), x);
    } else {
      const u32x4_t x = ld16(a.new_kv_c + tok * 1024 + lane * 16), y = ld16(a.new_k_pe + tok * 128 + (lane & 7) * 16);
      char* row = page + ((int64_t)scalar_load_i32(pages + slot) * P + (pos - slot * P)) * a.row_stride * 2;
      st16(row + lane * 16, x);
      if (lane < 8) st16(row + a.rope_offset * 2 + lane * 16, y);
    }
  }
}

// ---- balanced plan (one row per sequence): the 32-token tiles of the whole batch, sequence by
// sequence and inside a sequence head group by head group, are dealt evenly to the workgroups;
// workgroup j takes tiles [j * pw, (j + 1) * pw).  Pieces that are whole rows are finished in
// place, cut ones (at most the first and the last of a workgroup) leave partial rows in the
// workspace slots 2j and 2j + 1 (128 heads each).
//
// Starting a piece is not free: 147 KB of queries and the first tiles have to arrive and the
// piece before it has to be written out -- 17 us on the DeepSeek-V3 batch, five tiles' worth, and
// a workgroup with three pieces finished 37 us after one with a single piece.  So the line the
// workgroups share is padded: every (row, head group) is preceded by `piece_pad` tiles that hold
// no work.  A workgroup that runs into a new row spends that much of its share on the way, which
// is what the switch costs it; one that starts in the middle of a row, like most, pays nothing
// extra -- every workgroup has one start of its own anyway.
__device__ __forceinline__ int mla_tiles(int kv_len, int window) {
  if (kv_len <= 0) return 0;
  const int t_lo = (window > 0) ? max(0, kv_len - window) : 0;
  return (kv_len - (t_lo & ~(kTok - 1)) + kTok - 1) / kTok;
}

// extent of a (row, head group) on the padded line
__device__ __forceinline__ int mla_extent(const MlaDecodeArgs& a, int kv_len) {
  const int nt = mla_tiles(kv_len, a.sm.window);
  return nt > 0 ? nt + a.piece_pad : 0;
}

__device__ __forceinline__ int mla_tiles_per_wg(const MlaDecodeArgs& a, int total) {
  const int even = (total + a.num_wgs - 1) / a.num_wgs;  // the grid has exactly num_wgs workgroups
  return max(a.forced_tiles_per_wg > 0 ? a.forced_tiles_per_wg : a.min_tiles_per_wg, even);
}

// a.siblings > 1: so many workgroups take the same share or piece, each for heads of its own.  They walk the same tokens at the same
// time, so they are neighbours on one XCD (every eighth workgroup) and find each other's tiles in its L2.
struct Sibling {
  int unit, of;  // which of a.siblings, which share or piece
};
__device__ __forceinline__ Sibling sibling(const MlaDecodeArgs& a) {
  const int b = blockIdx.x;
  if (a.siblings <= 1) return {0, b};
  const int q = b >> 3, s = q / a.siblings;
  return {q - s * a.siblings, s * 8 + (b & 7)};
}

// `segment(mr, head_base, t_lo, t_begin, t_end, dest)` runs one piece on the workgroup's LDS ring.
// PUTS: the new tokens go into the cache here, in front of the pieces (otherwise it is the segment's business).
template <bool FP8, bool PUTS, class Segment>
__device__ __forceinline__ void mla_balanced_body(const MlaDecodeArgs& a, Segment segment) {
  const int lane = threadIdx.x & 63;
  int wg = sibling(a).of;  // this workgroup's share of the line
  const int num_wgs = a.num_wgs;
  if (wg >= num_wgs) return;  // (siblings: the grid is whole eights)
  const int units = (a.Hq + 127) / 128;
#ifdef RPA_MLA_TRACE
  if (threadIdx.x == 0) rpa_mla_trace_buf[blockIdx.x & 1023][0][7] = wall_clock64();  // kernel entry
#endif
  // prefix sums of tiles over the sequences: every wave scans (the result is wave-uniform)
  int total = 0, seq = -1, seq_first = 0;
  {
    // first pass: total; second pass (below) locates this workgroup's first tile
    for (int s0 = 0; s0 < a.num_rows; s0 += 64) {
      const int s = s0 + lane;
      int nt = (s < a.num_rows) ? mla_extent(a, a.pt.kv_lens[s]) : 0;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) nt += __shfl_xor(nt, off);
      total += nt;
    }
    total = __builtin_amdgcn_readfirstlane(total) * units;
  }
  const int pw = mla_tiles_per_wg(a, total);
  // The shares of an XCD's workgroups (every eighth) one after the other on the line: a row's pieces then find its queries, 147 KB at 128 heads,
  // in one L2.  10 rows of 500..5000 tokens x 16 heads 20.5 -> 19.7 us, 64 of 2000..16000 127.5 -> 126.2, 20 of 1000..9000 x 128 heads 55.8 -> 54.7; 3
  // rows of 8000..16000 x 128 heads, 27 shares each, 38.1 against 38.9: not with fewer rows than XCDs.
  const int per_xcd = ((total + pw - 1) / pw + 7) >> 3;  // (at most num_wgs / 8: the shares are at most num_wgs)
  if (a.num_rows >= 8 && (num_wgs & 7) == 0) {
    if ((wg >> 3) >= per_xcd && wg != 0) return;  // (the first one also writes the prefix sums of no work)
    wg = (wg & 7) * per_xcd + (wg >> 3);
  }
  if (wg == 0 && threadIdx.x < 64) {
    int base = 0;
    for (int s0 = 0; s0 < a.num_rows; s0 += 64) {
      const int s = s0 + lane;
      const int nt = (s < a.num_rows) ? mla_extent(a, a.pt.kv_lens[s]) : 0;
      int incl = nt;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int n = __shfl_up(incl, off);
        if (lane >= off) incl += n;
      }
      if (s < a.num_rows) a.cu_tiles[s + 1] = base + incl;
      base += __builtin_amdgcn_readfirstlane(__shfl(incl, 63));
    }
    if (lane == 0) a.cu_tiles[0] = 0;
  }
  if ((int64_t)wg * pw >= total) return;
  int x = wg * pw;
  const int x_end = min(total, x + pw);
  {
    int base = 0;
    for (int s0 = 0; s0 < a.num_rows && seq < 0; s0 += 64) {
      const int s = s0 + lane;
      const int nt = (s < a.num_rows) ? mla_extent(a, a.pt.kv_lens[s]) : 0;
      int incl = nt;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int n = __shfl_up(incl, off);
        if (lane >= off) incl += n;
      }
      const uint64_t hit = __builtin_amdgcn_ballot_w64((base + incl) * units > x);
      if (hit != 0) {
        const int first = __builtin_ctzll(hit);
        seq = s0 + first;
        seq_first = __builtin_amdgcn_readfirstlane((base + __shfl(incl - nt, first)) * units);
      } else {
        base += __builtin_amdgcn_readfirstlane(__shfl(incl, 63));
      }
    }
    seq = __builtin_amdgcn_readfirstlane(seq);
  }
  int kv_len = scalar_load_i32(a.pt.kv_lens + seq);
  int nt = mla_tiles(kv_len, a.sm.window);
  const int pad = a.piece_pad;
  if (PUTS && a.new_kv_c) {  // the new tokens of the rows that end in this share, all of them in front of its first piece
    int s = seq, len = kv_len, from = seq_first, tiles = nt;
    for (;;) {
      const int unit_end = from + (max(x - from, 0) / (tiles + pad) + 1) * (tiles + pad);
      if (unit_end > x_end) break;
      put_new_row<FP8>(a, s, len);
      from += (tiles + pad) * units;
      if (from >= x_end) break;
      do {
        ++s;
        len = scalar_load_i32(a.pt.kv_lens + s);
        tiles = mla_tiles(len, a.sm.window);
      } while (tiles == 0);
    }
    wait_all_loads();  // (and stores)
  }
  bool first_piece = true;
  int piece_no = 0;  // (only the optional timestamps use it)
  while (x < x_end) {
    const int r = x - seq_first;  // position inside the row's padded extents
    const int unit = r / (nt + pad);
    int off = r - unit * (nt + pad);
    if (off < pad) {  // the padding in front of this (row, head group): no work there
      x += pad - off;
      off = pad;
      if (x >= x_end) break;
    }
    const int tile = off - pad;
    const int take = min(nt - tile, x_end - x);
    const int t_lo = (a.sm.window > 0) ? max(0, kv_len - a.sm.window) : 0;
    const int t0 = t_lo & ~(kTok - 1);
    MlaRow mr;
    mr.seq = seq;
    mr.kv_len = kv_len;
    mr.tq = scalar_load_i32(a.pt.cu_q_lens + seq);
    mr.valid = true;
    MlaDest dest;
    dest.final_rows = (tile == 0) && (take == nt);
    dest.base = ((int64_t)wg * 2 + (first_piece ? 0 : 1)) * 128 - unit * 128;  // + head
    first_piece = false;
    segment(mr, unit * 128, t_lo, t0 + tile * kTok, min(kv_len, t0 + (tile + take) * kTok), dest, piece_no++);
    x += take;
    if (x < x_end && tile + take == nt && unit == units - 1) {
      seq_first += (nt + pad) * units;
      do {
        ++seq;
        kv_len = scalar_load_i32(a.pt.kv_lens + seq);
        nt = mla_tiles(kv_len, a.sm.window);
      } while (nt == 0);
    }
  }
}

}  // namespace
}  // namespace rpa
