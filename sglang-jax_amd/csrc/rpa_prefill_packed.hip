// Flash kernel for prefill launches that the tiles of 128 query positions leave mostly idle on gfx950: one prompt on a
// tensor-parallel share of the heads, a few short chunks, a verify step of speculative decoding.
//
// What bounds such a launch is a chain: a workgroup of rpa_prefill_pipe_kernel walks its 64-token K/V tiles one after the
// other, 16 of them for a prompt of 1003 tokens, about 1 us each, on 64 of 256 CUs.  Here a workgroup owns 32 COLUMNS and
// its eight waves walk DIFFERENT tiles:
//   * a column is a (query position, query head) pair: the G query heads of a kv head times 32 / G positions, so that the
//     32-column matrix instructions are full also for a chunk of a few tokens, and a kv head's rows are read once for all
//     of its query heads (a verify step of 8 tokens on 2 heads per kv head has 16 columns; the 128-position tile ran it on
//     8 rows of 128)
//   * wave w takes the 32-token tiles w, w + 8, ...: a chain of 4 instead of 16 for 1003 tokens, and no barrier in it (every
//     wave copies its own tiles into its own LDS).  The eight partial results meet in LDS at the end, in f32.
// The price is that K/V rows are brought into LDS once per 32 columns instead of once per 128 (64 B per clock and CU from the
// L2: 4 us for the 512 KB of the longest workgroup of that prompt), so launches that fill the GPU stay where they were:
// see prefill_packed_pieces().
//
// A wave's tile, single buffers: K of the next tile is requested when this tile's scores have been taken, V when its second
// product has; each copy then has the other half of the step to arrive.  bf16 rows: LDS layout and swizzles of
// rpa_prefill_async_kernel.  e4m3 rows arrive as bytes; K operands are widened on their way from LDS to the matrix pipe, V
// rows into a bf16 tile for the transposing reads.

#include <cmath>
#include <type_traits>

#include "rpa_prefill_common.h"

namespace rpa {

using namespace pf;

namespace {

constexpr int kWaves = 8;
constexpr int kTok = 32;                  // tokens per tile
constexpr int kCols = 32;                 // (position, head) pairs per workgroup
constexpr int kFeedB = 16384;             // LDS of a wave: bf16 K, V; e4m3 K bytes, V bytes, V widened
constexpr int kMergePitch = 132;          // floats per column in the merge (16-byte writes of 16 columns meet every bank once)
constexpr int kMergeB = kWaves * kCols * kMergePitch * 4;
constexpr int kIdsAt = kWaves * kFeedB;   // 64 page ids per wave
constexpr int kMaskPairs = 8;             // pairs of mask rows per workgroup (two query heads per kv head and more)
constexpr int kMaskB = kMaskPairs * 256;  // of a wave: 32 words of two rows per copy instruction
constexpr int kMaskAt = kIdsAt + kWaves * 256;
constexpr int kMlAt = kMaskAt + kWaves * kMaskB;
constexpr int kLdsB = kMlAt + kWaves * kCols * 8;
static_assert(kMergeB <= kMlAt, "the merge reuses the tiles, not the (maximum, sum) pairs");

typedef __attribute__((address_space(3))) char* lds_t;
typedef float f32x4v_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xC07F); }  // lgkmcnt(0)

// PG: pages of a tile.  1: the tile lies inside a page (page size a multiple of 32); 2: pages of 16 tokens; 0: any other
// size, page ids through LDS (a load into a register would make the compiler drain the copies in flight).
// SGPR_BACK: the kernel has so many scalars that the compiler keeps a tile's base in vector registers from one copy to the next.
template <int PG, bool FP8, bool SGPR_BACK>
struct PackedFeed {
  static constexpr int kPerRow = FP8 ? 8 : 16;        // 16-byte chunks of a row of 128 elements
  static constexpr int kRowsPer = 64 / kPerRow;       // rows per copy instruction
  static constexpr int N = kTok / kRowsPer;           // copy instructions for the K (or V) rows of a tile
  static constexpr int kTileBytes = N * 1024;

  uint32_t ofs_k[N], ofs_v[N];  // a lane's chunk from the first row of its page part (PG 2: 16 rows) of a whole tile
  int64_t base[PG == 2 ? 2 : 1];  // byte offset of the tile's first row(s), the same in every lane
  int64_t row[N];               // PG 0: per-lane byte offsets of the rows
  uint32_t fresh;               // PG 0, bit n: this lane's row of copy n is a new token's (row[n] counts from the caller's rows then)
  bool whole;
  int first, last;              // the tile's first token, the sequence's last
  // New tokens that are not in the cache yet: those from position new_from on, new_stride bytes apart in the caller's rows.
  int new_from, new_stride;

  __device__ __forceinline__ static int row_of(int n, int lane) { return n * kRowsPer + lane / kPerRow; }
  __device__ __forceinline__ static int chunk_k(int t, int cp) { return FP8 ? cp ^ ((t >> 1) & 7) : cp ^ (t & 15); }
  __device__ __forceinline__ static int chunk_v(int t, int cp) { return FP8 ? cp : cp ^ ((t & 3) << 2); }

  __device__ __forceinline__ void init(const KvAddr& kv, int lane) {
    const int cp = lane % kPerRow;
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int t = row_of(n, lane), in = PG == 2 ? (t & 15) : t;
      ofs_k[n] = (uint32_t)(in * kv.tok_stride + (chunk_k(t, cp) << 4));
      ofs_v[n] = (uint32_t)(in * kv.tok_stride + (chunk_v(t, cp) << 4));
    }
  }

  __device__ __forceinline__ static void request_ids(uint32_t at, const TileSrc& s, int tb, int lane) {
    tb = min(tb, s.last_tok);
    const int32_t* src = s.pages + min(page_slot(s, tb) + lane, page_slot(s, s.last_tok));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(at), "v"(src) : "memory", "m0");
  }

  // Where the rows of the tile at `tb` are (PG 0: its page ids have arrived at `ids`).
  __device__ __forceinline__ void locate(const TileSrc& s, const KvAddr& kv, int tb, int lane, uint32_t ids) {
    whole = PG != 0 && tb + kTok - 1 <= min(s.last_tok, new_from - 1);
    first = tb;
    last = s.last_tok;
    if constexpr (PG == 0) {
#pragma unroll
      for (int n = 0; n < N; ++n) {
        const int tok = min(tb + row_of(n, lane), s.last_tok), ps = page_slot(s, tok);
        const int id = *(__attribute__((address_space(3))) const int32_t*)(lds_t)(uintptr_t)(ids + 4u * (uint32_t)(ps - page_slot(s, tb)));
        row[n] = (int64_t)id * kv.page_stride + (int64_t)(tok - ps * s.page_size) * kv.tok_stride;
      }
      fresh = 0;
      if (tb + kTok > new_from) {  // (the same in every lane)
#pragma unroll
        for (int n = 0; n < N; ++n) {
          const int past = min(tb + row_of(n, lane), s.last_tok) - new_from;
          if (past >= 0) {
            row[n] = (int64_t)past * new_stride;
            fresh |= 1u << n;
          }
        }
      }
    } else {
      const int ps = __builtin_amdgcn_readfirstlane(page_slot(s, tb));
      const int pg0 = scalar_load_i32(s.pages + ps);
      const int pg1 = PG == 2 ? scalar_load_i32(s.pages + min(ps + 1, page_slot(s, s.last_tok))) : pg0;
      base[0] = (int64_t)pg0 * kv.page_stride + (PG == 1 ? (int64_t)(tb - ps * s.page_size) * kv.tok_stride : 0);
      if constexpr (PG == 2) base[1] = (int64_t)pg1 * kv.page_stride;
    }
  }

  template <bool IS_V>
  __device__ __forceinline__ void copy(uint32_t at, const KvAddr& kv, const char* head, const char* new_head, int lane) const {
    if (PG != 0 && first + kTok <= new_from) {
      auto put = [&](int n, uint32_t o, const char* b) __attribute__((always_inline)) {
        if constexpr (SGPR_BACK) {  // (the wait: see async_copy16_from)
          const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)b), hi = __builtin_amdgcn_readfirstlane((uint32_t)((uintptr_t)b >> 32));
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(at + n * 1024), "v"(o), "s"(((uint64_t)hi << 32) | lo) : "memory", "m0");
        } else {
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(at + n * 1024), "v"(o), "s"(b) : "memory", "m0");
        }
      };
      if (whole) {
#pragma unroll
        for (int n = 0; n < N; ++n) put(n, IS_V ? ofs_v[n] : ofs_k[n], head + base[PG == 2 && n >= N / 2 ? PG - 1 : 0]);
      } else {  // the sequence's last tile: rows behind its end repeat the last one
        const int end = last - first;
        const bool upper = PG == 2 && end >= 16;
#pragma unroll
        for (int n = 0; n < N; ++n) {
          const int row = row_of(n, lane), own = PG == 2 ? (row & 15) : row;  // from the row that the copy's offsets count from
          const int to = PG == 2 && n >= N / 2 && upper ? min(own, end - 16) : min(row, end);
          put(n, (IS_V ? ofs_v[n] : ofs_k[n]) - (uint32_t)((own - to) * kv.tok_stride), head + base[PG == 2 && n >= N / 2 && upper ? PG - 1 : 0]);
        }
      }
    } else if constexpr (PG != 0) {
      // Tiles with new tokens, an address per lane: few, so what they take is not unrolled into the loop around it (with an address per row and
      // copy kept, that grew by a third and its scalars went to vector registers and back).
      const int cp = lane % kPerRow;
      int64_t b0 = base[0], b1 = base[PG == 2 ? 1 : 0];
      asm volatile("" : "+v"(b0), "+v"(b1));  // (the bases themselves have to stay scalars)
#pragma unroll 1
      for (int n = 0; n < N; ++n) {
        const int in = row_of(n, lane), t = min(in, last - first), past = first + t - new_from;
        const int64_t old = PG == 2 ? (t >= 16 ? b1 : b0) + (int64_t)((t & 15) * kv.tok_stride) : b0 + (int64_t)(t * kv.tok_stride);
        const char* g = (past >= 0 ? new_head + (int64_t)past * new_stride : head + old) + ((IS_V ? chunk_v(in, cp) : chunk_k(in, cp)) << 4);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(at + n * 1024), "v"(g) : "memory", "m0");
      }
    } else {
      const int cp = lane % kPerRow;
      auto put = [&](int n, const char* from) __attribute__((always_inline)) {
        const int t = row_of(n, lane);
        const char* g = from + row[n] + ((IS_V ? chunk_v(t, cp) : chunk_k(t, cp)) << 4);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(at + n * 1024), "v"(g) : "memory", "m0");
      };
      if (first + kTok <= new_from) {
#pragma unroll
        for (int n = 0; n < N; ++n) put(n, head);
      } else {
#pragma unroll
        for (int n = 0; n < N; ++n) put(n, (fresh >> n) & 1 ? new_head : head);
      }
    }
  }
};

__device__ __forceinline__ u32x4_t at16(uint32_t at) {
  return *(__attribute__((address_space(3))) const u32x4_t*)(lds_t)(uintptr_t)at;
}
__device__ __forceinline__ u32x2_t at8(uint32_t at) {
  return *(__attribute__((address_space(3))) const u32x2_t*)(lds_t)(uintptr_t)at;
}
__device__ __forceinline__ u32x2_t at_tr(uint32_t at) {
  typedef __attribute__((address_space(3))) s16x4_t* ptr_t;
  return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr_t)(uintptr_t)at));
}

// soft cap, temperature and rounding of 16 scores, to log2 units (as softmax_tile has them)
template <class Smx>
__device__ __forceinline__ void general_scores(f32x16_t& S, const Smx& sm) {
  if (sm.cap != 0.f && !sm.round_mode) {
    const float k1 = sm.scale * sm.inv_cap * (2.0f * kLog2e), k2 = sm.cap * sm.temp * kLog2e;
#pragma unroll
    for (int v = 0; v < 16; ++v) S[v] = __builtin_fmaf(__builtin_amdgcn_rcpf(fast_exp2(S[v] * k1) + 1.0f), -2.0f * k2, k2);
  } else {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      float x = S[v] * sm.scale;
      if (sm.cap != 0.f) x = soft_cap_f(x, sm.cap, sm.inv_cap);
      x = x * sm.temp;
      if (sm.round_mode) x = round_logit(x, sm.round_mode);
      S[v] = x * kLog2e;
    }
  }
}

// grid: (sequence, kv head) units x tiles of `per` = 32 / G positions, then the workgroups that write a prompt's rows;
// blockIdx.y = piece of the K/V range.  CAP: soft cap or rounded logits; EXT: custom or no mask, temperature, q_scale.
// WORDS: custom mask, read as the caller has it: a wave copies the 32 words of its tile of every mask row that it has columns of,
// two rows to an instruction, and a ballot makes bits of them.  (Bits made by a launch of their own in front cost that launch, and the
// general masked path loads a word per score where there are none: a verify step is a handful of rows, 12 % of what its K/V rows are.)
//
// New tokens (a.tail_is_new): a verify step or a short chunk had a launch in front that put its tokens into the cache, and read them from there.
// Tiles with new tokens take those rows from the caller's, an address per lane; workgroups behind the attention's write the cache.
// With both, us of the call: 2 verify steps of 4 tokens on 222..1322 x 8 / 4 heads 18.4 -> 11.0, x 32 / 8 19.0 -> 11.9, 8 of 8 on 3800..7600 x 16 / 8 50.5 ->
// 39.8, 16 of 4 on 1000..7000 x 32 / 8 75.9 -> 49.9 (162 drawn steps 1.58 x, with what moved here from other kernels); chunks of 69 tokens on 760 x 8 / 4
// heads 18.0 -> 11.6, of 110 in all on 1400 x 8 / 1 19.5 -> 13.8.
template <int PG, bool CAP, bool EXT, bool FP8, bool WORDS = false>
__global__ __launch_bounds__(512, 2) void rpa_prefill_packed_kernel(const PrefillArgs a_in, int tiles, int nseq, int per) {
  static_assert(!WORDS || (EXT && !CAP), "words of a mask come without other options");
  PrefillArgs a = a_in;  // static-shape mode: the sequences to process come from the device
  if (a.dist) {
    a.seq_begin = (a.sm.mask_mode == 1) ? 0 : scalar_load_i32(a.dist);
    a.seq_end = min(a.seq_end, scalar_load_i32(a.dist + 2));
  }
  __shared__ __attribute__((aligned(1024))) char lds[kLdsB];
  // where a sequence's mask rows begin, if the caller does not say: words of the sequences in front of it, one per lane, asked for with
  // everything else that a workgroup looks up
  int mask_rows = 0, mask_width = 0;
  auto mask_of = [&](int s) __attribute__((always_inline)) {
    mask_rows = a.pt.cu_q_lens[s + 1] - a.pt.cu_q_lens[s];
    mask_width = a.sm.mask_rows_page_aligned ? a.pt.cu_kv_lens[s + 1] - a.pt.cu_kv_lens[s] : a.pt.kv_lens[s];
  };
  if constexpr (WORDS) {
    const int s = a.seq_begin + (int)(threadIdx.x & 63);
    if (!a.sm.cu_mask_lens && s < a.seq_end) mask_of(s);
  }
  const Work w = decompose(a, tiles, nseq, false, per, a.G);
  if (__builtin_expect(!w.valid, 0)) {
    write_tail_tokens(a_in);
    return;
  }
  typedef PackedFeed<PG, FP8, WORDS> Feed;
  constexpr int N = Feed::N;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 31, h = lane >> 5;
  const TileSrc src = make_src(a, w);
  const char* kh = head_rows(a, w, a.kv.k_base);
  const char* vh = head_rows(a, w, a.kv.v_base);
  const int new_stride = a.Hkv * (kHeadDim * (FP8 ? 1 : 2));
  const int64_t new_at = a.tail_is_new ? (int64_t)w.qg0 * new_stride + w.hk * (kHeadDim * (FP8 ? 1 : 2)) : 0;
  const char *new_k = a.write.keys + new_at, *new_v = a.write.values + new_at;

  // columns: position c / G, head c % G; those behind the last whole position, and positions past the chunk, are not written
  const int r_lo = w.q_start, r_hi = min(w.q_start + per, w.q_len) - 1;
  const int pos = c / a.G;
  const int row = r_lo + pos, qpos = w.prefix + row;
  const int W_ = a.sm.window;
  const bool causal = !WORDS && (!EXT || a.sm.mask_mode == 0);
  MaskCtx mc;
  mc.mode = 0;
  if constexpr (WORDS) {
    mc.mode = 1;
    mc.kv_len = w.kv_len;
  } else if constexpr (EXT) {
    mc = make_mask_ctx(a, w, min(row, r_hi));
  }
  int t_hi = causal ? min(w.kv_len, w.prefix + r_hi + 1) : w.kv_len;  // exclusive
  int t_lo = 0;
  if (W_ > 0) t_lo = max(0, w.prefix + r_lo - W_ + 1) & ~(kBN - 1);
  int split = 0;
  if (a.kv_splits > 1 && !kv_piece(a, t_lo, t_hi, split)) t_hi = t_lo;  // nothing left for this piece: rows that weigh nothing
  t_lo = __builtin_amdgcn_readfirstlane(t_lo);
  t_hi = __builtin_amdgcn_readfirstlane(t_hi);
  const int nT = max(0, (t_hi - t_lo + kTok - 1) / kTok);

  const uint32_t lds_at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_t)lds);
  const uint32_t k_at = lds_at + wave * kFeedB, v_at = k_at + Feed::kTileBytes;
  const uint32_t vt_at = FP8 ? k_at + 2 * Feed::kTileBytes : v_at;  // V rows as bf16
  const uint32_t ids_at = lds_at + kIdsAt + wave * 256, mask_at = lds_at + kMaskAt + wave * kMaskB;
  const bool has_bits = EXT && !WORDS && mc.mode == 1 && mc.bits;  // (else the caller's words, one load per score)
  // Columns that are not written see what the last row does: all columns of a wave have their references raised together, so what any of them sees is
  // part of how the others' probabilities are rounded (and nothing may depend on what LDS holds behind the rows that were copied).
  const int mask_row = min(pos, r_hi - r_lo);
  const int my_rows = r_hi - r_lo + 1, pairs = WORDS ? __builtin_amdgcn_readfirstlane((my_rows + 1) >> 1) : 0;
  uint64_t mask = 0;   // WORDS: this workgroup's first row
  uint32_t pitch = 0;  // bytes of a row
  if constexpr (WORDS) {
    int64_t first = 0;
    const int width = a.sm.mask_rows_page_aligned ? scalar_load_i32(a.pt.cu_kv_lens + w.seq + 1) - scalar_load_i32(a.pt.cu_kv_lens + w.seq) : w.kv_len;
    if (a.sm.cu_mask_lens) {
      first = scalar_load_i32(a.sm.cu_mask_lens + w.seq);
    } else {
      for (int s = a.seq_begin + lane; s < w.seq; s += 64) {
        if (s >= a.seq_begin + 64) mask_of(s);
        first += (int64_t)mask_rows * mask_width;
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) first += __shfl_xor(first, off);
    }
    const uint64_t at = reinterpret_cast<uint64_t>(a.sm.custom_mask + first + (int64_t)r_lo * width);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)at), hi = __builtin_amdgcn_readfirstlane((uint32_t)(at >> 32));
    mask = ((uint64_t)hi << 32) | lo;
    pitch = __builtin_amdgcn_readfirstlane(4 * width);
  }
  auto request_mask = [&](int tb) __attribute__((always_inline)) {
    if constexpr (WORDS) {  // (tokens from kv_len on are masked in any case)
      const uint32_t in_row = 4u * (uint32_t)min(lane & 31, w.kv_len - 1 - tb), upper = in_row + (lane >> 5) * pitch;
      const uint64_t words = mask + 4u * (uint32_t)tb;
#pragma unroll
      for (int i = 0; i < kMaskPairs; ++i) {
        if (i < pairs) {  // (an odd last row stands for the one behind it; the wait: see async_copy16_from)
          asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 3\n\tglobal_load_lds_dword %2, %3"
                       ::"s"(mask_at), "n"(i * 256), "v"(2 * i + 1 < my_rows ? upper : in_row), "s"(words + (uint64_t)(2 * i) * pitch) : "memory", "m0", "scc");
        }
      }
    } else {
      const uint32_t* words = reinterpret_cast<const uint32_t*>(mc.bits) + min(tb >> 5, 2 * mc.bit_words - 1);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(mask_at), "v"(words) : "memory", "m0");
    }
  };
  const bool has_mask = WORDS || has_bits;
  // V's copies have landed; those of the next tile's K, and of its mask behind them, may be on their way
  auto wait_v = [&]() __attribute__((always_inline)) {
    if (!has_mask) __builtin_amdgcn_s_waitcnt(0x0F70 | N);
    else if (!WORDS || pairs < 2) __builtin_amdgcn_s_waitcnt(0x0F70 | (N + 1));
    else if (pairs < 4) __builtin_amdgcn_s_waitcnt(0x0F70 | (N + 2));
    else __builtin_amdgcn_s_waitcnt(0x0F70 | (N + 4));
  };

  Feed feed;
  feed.new_from = a.tail_is_new ? w.prefix : 0x7fffffff;
  feed.new_stride = new_stride;
  int j = wave;  // this wave's tile
  if (j < nT) {
    const int tb = t_lo + j * kTok;
    if constexpr (PG == 0) {
      Feed::request_ids(ids_at, src, tb, lane);
      wait_all_loads();
    }
    feed.init(a.kv, lane);
    feed.locate(src, a.kv, tb, lane, ids_at);
    if constexpr (PG == 0) {
      wait_lds();
      Feed::request_ids(ids_at, src, tb + kWaves * kTok, lane);
    }
    feed.template copy<false>(k_at, a.kv, kh, new_k, lane);
    if (has_mask) request_mask(tb);
    feed.template copy<true>(v_at, a.kv, vh, new_v, lane);
  }

  u32x4_t qB[kSteps];
  {
    const int head = w.head + (c - pos * a.G);
    const uint16_t* qp = a.q + ((int64_t)(w.qg0 + min(row, w.q_len - 1)) * a.Hq + head) * a.q_dim;
    ld_query_row<kSteps, kHeadDim>(qB, qp, h, a.q_dim);
    if (EXT && !WORDS && a.sm.q_scale > 0.f) {
#pragma unroll
      for (int ks = 0; ks < kSteps; ++ks) qB[ks] = requantise_q(qB[ks], a.sm.q_scale, FP8);
    }
  }
  Softmax<CAP> sm;
  sm.scale = a.sm.sm_scale * (a.k_scale ? scalar_load_f32(a.k_scale + w.hk) : 1.0f) *
             ((EXT && !WORDS && a.sm.q_scale > 0.f) ? a.sm.q_scale : 1.0f);
  make_scale_positive(sm.scale, qB);
  sm.cap = a.sm.soft_cap;
  sm.inv_cap = (sm.cap != 0.f) ? 1.0f / sm.cap : 0.f;
  {
    const float temp = EXT && !WORDS ? xai_factor(qpos, a.sm.xai_len) : 1.0f;  // per query position
    sm.sc2 = CAP ? 1.0f : sm.scale * kLog2e * temp;
    sm.temp = temp;
    sm.round_mode = a.sm.round_logits;
  }

  f32x16_t O[kDimTiles];
#pragma unroll
  for (int d = 0; d < kDimTiles; ++d) O[d] = kZero16;
  float m = kMaxFloor, l = 0.f;

  // operand addresses inside a tile: see rpa_prefill_async_kernel
  uint32_t koff[kSteps], voff[kDimTiles];
  {
    const int r16 = lane & 15, b16 = lane >> 4;
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks)
      koff[ks] = FP8 ? k_at + c * 128 + ((ks ^ ((c >> 1) & 7)) << 4) + 8 * h : k_at + c * kRowB + ((ks * 32) ^ ((h ^ (c & 15)) << 4));
#pragma unroll
    for (int d = 0; d < kDimTiles; ++d)
      voff[d] = vt_at + (4 * h + (r16 >> 2)) * kRowB + ((b16 & 1) << 5) + (((r16 & 3) >> 1) << 4) + ((r16 & 1) << 3) + ((d * 64) ^ ((r16 >> 2) << 6));
  }
  const bf16x2_t ones = {(__bf16)1.0f, (__bf16)1.0f};

  while (j < nT) {
    const int tb = t_lo + j * kTok;
    const bool more = j + kWaves < nT;
    __builtin_amdgcn_s_waitcnt(0x0F70 | N);  // K has landed (V's copies are younger)
    asm volatile("" ::: "memory");
    uint32_t mask_word = 0;
    if constexpr (WORDS) {
      auto take = [&](auto tag) __attribute__((always_inline)) {
        int x[decltype(tag)::value];
#pragma unroll
        for (int i = 0; i < decltype(tag)::value; ++i)
          x[i] = *(__attribute__((address_space(3))) const int32_t*)(lds_t)(uintptr_t)(mask_at + i * 256 + 4u * lane);
#pragma unroll
        for (int i = 0; i < decltype(tag)::value; ++i) {
          const uint64_t keep = __ballot(x[i] >= 1);
          const uint32_t mine = (mask_row & 1) ? (uint32_t)(keep >> 32) : (uint32_t)keep;
          mask_word = (mask_row >> 1) == i ? mine : mask_word;
        }
      };
      if (pairs <= 2) take(std::integral_constant<int, 2>{});
      else if (pairs <= 4) take(std::integral_constant<int, 4>{});
      else take(std::integral_constant<int, kMaskPairs>{});
    }
    if (has_bits) mask_word = *(__attribute__((address_space(3))) const uint32_t*)(lds_t)(uintptr_t)(mask_at + 4u * lane);
    f32x16_t S = kZero16;
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks) {
      if constexpr (FP8) {
        const u32x2_t x = at8(koff[ks]);
        const u32x2_t lo = fp8x4_to_bf16x4(x[0]), hi = fp8x4_to_bf16x4(x[1]);
        S = mfma32(u32x4_t{lo[0], lo[1], hi[0], hi[1]}, qB[ks], S);
      } else {
        S = mfma32(at16(koff[ks]), qB[ks], S);
      }
    }
    if (more) {
      const int tn = tb + kWaves * kTok;
      feed.locate(src, a.kv, tn, lane, ids_at);
      wait_lds();  // the reads of K (and of the ids and the mask) have returned: their places may be filled again
      if constexpr (PG == 0) Feed::request_ids(ids_at, src, tn + kWaves * kTok, lane);
      feed.template copy<false>(k_at, a.kv, kh, new_k, lane);
      if (has_mask) request_mask(tn);
    }

    // ---- softmax of the 16 scores of this lane: tokens tb + 8 (v / 4) + 4 h + v % 4
    if constexpr (CAP) general_scores(S, sm);
    const bool need_mask = (causal ? (tb + kTok - 1 > w.prefix + r_lo) : (mc.mode == 1 || tb + kTok > w.kv_len)) ||
                           (W_ > 0 && tb <= w.prefix + r_hi - W_);
    if (WORDS || has_bits) {
      // what the row may see as bits: the caller's mask, tokens of the sequence, the window
      const int end = w.kv_len - tb, from = W_ > 0 ? qpos - W_ + 1 - tb : 0;
      mask_word &= end < 32 ? (1u << end) - 1u : ~0u;
      if (from > 0) mask_word &= from < 32 ? ~0u << from : 0u;
      mask_word >>= 4 * h;
#pragma unroll
      for (int v = 0; v < 16; ++v) S[v] = (mask_word >> (8 * (v >> 2) + (v & 3))) & 1u ? S[v] : kMaskRaw;
    } else if (need_mask) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int tok = tb + 8 * (v >> 2) + 4 * h + (v & 3);
        bool masked;
        if (!EXT || mc.mode == 0) masked = tok > qpos;
        else masked = (tok >= mc.kv_len) || (mc.mode == 1 && mc.row[tok] < 1);
        masked = masked || (W_ > 0 && tok <= qpos - W_);
        S[v] = masked ? kMaskRaw : S[v];
      }
    }
    float mx = __builtin_fmaxf(S[0], S[1]);
#pragma unroll
    for (int v = 2; v < 16; v += 2) mx = __builtin_fmaxf(__builtin_fmaxf(mx, S[v]), S[v + 1]);
    update_running_max(swap_max(mx), m, l, O, sm.sc2);
    const float neg_m = -m * sm.sc2;
    u32x4_t pB[2];
    float ps[2] = {0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t x = pack_bf16x2(fast_exp2(__builtin_fmaf(S[2 * i], sm.sc2, neg_m)), fast_exp2(__builtin_fmaf(S[2 * i + 1], sm.sc2, neg_m)));
      ps[i & 1] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, x), ones, ps[i & 1], false);
      pB[i >> 2][i & 3] = x;
    }
    l += ps[0] + ps[1];

    if (more) wait_v();
    else __builtin_amdgcn_s_waitcnt(0x0F70);
    asm volatile("" ::: "memory");
    if constexpr (FP8) {  // bytes -> bf16 rows, two chunks of 16 bytes each
#pragma unroll
      for (int n = 0; n < N; ++n) {
        const int t = Feed::row_of(n, lane), cp = 2 * (lane & 7);
        const u32x4_t x = at16(v_at + n * 1024 + lane * 16);
        const u32x2_t p = fp8x4_to_bf16x4(x[0]), q = fp8x4_to_bf16x4(x[1]), r = fp8x4_to_bf16x4(x[2]), s = fp8x4_to_bf16x4(x[3]);
        const uint32_t at = vt_at + t * kRowB;
        *(__attribute__((address_space(3))) u32x4_t*)(lds_t)(uintptr_t)(at + ((cp ^ ((t & 3) << 2)) << 4)) = u32x4_t{p[0], p[1], q[0], q[1]};
        *(__attribute__((address_space(3))) u32x4_t*)(lds_t)(uintptr_t)(at + (((cp + 1) ^ ((t & 3) << 2)) << 4)) = u32x4_t{r[0], r[1], s[0], s[1]};
      }
      wait_lds();
      asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int d = 0; d < kDimTiles; ++d) {
        const u32x2_t lo = at_tr(voff[d] + kk * 16 * kRowB), hi = at_tr(voff[d] + kk * 16 * kRowB + 8 * kRowB);
        O[d] = mfma32(u32x4_t{lo[0], lo[1], hi[0], hi[1]}, pB[kk], O[d]);
      }
    if (more) {
      wait_lds();
      feed.template copy<true>(v_at, a.kv, vh, new_v, lane);
    }
    j += kWaves;
  }

  // ---- merge of the waves' results, in f32: references and sums first, then the rows against the largest reference
  typedef __attribute__((address_space(3))) f32x2_t* ml_t;
  const uint32_t ml_at = lds_at + kMlAt;
  l += __shfl_xor(l, 32);
  const float m2 = wave < nT ? fmaxf(m * sm.sc2, kNoReference) : kNoReference;
  if (h == 0) *(ml_t)(uintptr_t)(ml_at + (wave * kCols + c) * 8) = f32x2_t{m2, l};
  __syncthreads();
  const int n_waves = min(nT, kWaves);  // waves that had a tile
  auto reference = [&](int col, float& den) __attribute__((always_inline)) {
    f32x2_t x[kWaves];
    float top = kNoReference;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) {
      x[i] = *(ml_t)(uintptr_t)(ml_at + (i * kCols + col) * 8);
      top = fmaxf(top, x[i][0]);
    }
    den = 0.f;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) den += x[i][1] * fast_exp2(x[i][0] - top);
    return top;
  };
  float den;
  if (wave < nT) {
    const float f = fast_exp2(m2 - reference(c, den));
    typedef __attribute__((address_space(3))) f32x4v_t* o_t;
    const uint32_t at = lds_at + ((wave * kCols + c) * kMergePitch + 4 * h) * 4;
#pragma unroll
    for (int d = 0; d < kDimTiles; ++d)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *(o_t)(uintptr_t)(at + (d * 32 + q * 8) * 4) = f32x4v_t{O[d][4 * q] * f, O[d][4 * q + 1] * f, O[d][4 * q + 2] * f, O[d][4 * q + 3] * f};
  }
  __syncthreads();
  const int col = threadIdx.x >> 4, dim = (threadIdx.x & 15) * 8;
  const int out_pos = col / a.G, out_row = r_lo + out_pos, head = w.head + col - out_pos * a.G;
  if (out_pos >= per || out_row >= w.q_len) return;
  const float top = reference(col, den);
  float o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = 0.f;
  for (int i = 0; i < n_waves; ++i) {
    typedef __attribute__((address_space(3))) const f32x4v_t* o_t;
    const uint32_t at = lds_at + ((i * kCols + col) * kMergePitch + dim) * 4;
    const f32x4v_t x = *(o_t)(uintptr_t)at, y = *(o_t)(uintptr_t)(at + 16);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] += x[e];
      o[4 + e] += y[e];
    }
  }
  const int64_t out_at = (int64_t)(w.qg0 + out_row) * a.Hq + head;
  if (a.kv_splits > 1) {
    const int64_t slot = out_at * a.kv_splits + split;
    float* op = a.ws_o + slot * kHeadDim + dim;
    *reinterpret_cast<f32x4v_t*>(op) = f32x4v_t{o[0], o[1], o[2], o[3]};
    *reinterpret_cast<f32x4v_t*>(op + 4) = f32x4v_t{o[4], o[5], o[6], o[7]};
    if (dim == 0) {
      a.ws_ml[slot * 2] = top;
      a.ws_ml[slot * 2 + 1] = den;
    }
    return;
  }
  if (dim >= a.q_dim) return;
  const float vs = a.v_scale ? scalar_load_f32(a.v_scale + w.hk) : 1.0f;
  const float inv = a.sm.sink ? vs * sink_inverse(top, den, sink_logit(a.sm.sink, a.sm.round_logits, head)) : vs / den;
  st16(a.out + out_at * a.q_dim + dim, u32x4_t{pack_bf16x2(o[0] * inv, o[1] * inv), pack_bf16x2(o[2] * inv, o[3] * inv),
                                               pack_bf16x2(o[4] * inv, o[5] * inv), pack_bf16x2(o[6] * inv, o[7] * inv)});
}

}  // namespace

// Microseconds of a launch with every K/V range in n pieces, fitted to 60 prompts, chunks and verify steps of 8 .. 2048
// tokens on prefixes of 0 .. 16384 (both kernels).  A workgroup has a CU to itself and pays 4.5 us (custom masks: 5.5 as words, 6.5 as bits) for its
// start and its merge; eight tiles side by side take 1.25 us of a lone workgroup, up to 1.1 us more where few workgroups read the same
// rows (they come from HBM), 1.45 us on a full chip; workgroups of the grid that find no tile 0.4 us a round; pieces the merge launch and the partial rows' way to memory and
// back.
static double packed_us(const PrefillArgs& a, int nseq, int n) {
  const int per = kCols / a.G;
  const int64_t tokens = std::max<int64_t>(1, (int64_t)a.num_tokens - a.seq_begin);
  const int64_t grid = (int64_t)nseq * ((a.max_q_len + per - 1) / per) * a.Hkv;
  const int64_t wgs = std::min(grid, (tokens / per + nseq) * a.Hkv);
  double longest = a.max_kv_len, mean = std::max(1.0, a.max_kv_len - 0.5 * (a.max_q_len - 1));
  if (a.sm.window > 0) {
    longest = std::min(longest, (double)a.sm.window + per + kBN);
    mean = std::min(mean, longest);
  }
  auto steps = [&](double range) { return std::ceil(std::ceil(range / n / kTok) / kWaves); };
  const double step_us = 1.25 + 1.1 / ((a.max_q_len + per - 1) / per), start_us = a.sm.mask_mode != 1 ? 4.5 : a.mask_words ? 5.5 : 6.5;
  const double cus = compute_units(), rounds = std::ceil((double)wgs * n / cus);
  const double full = rounds * start_us + 1.45 * (double)wgs * n * steps(mean) / cus + 0.4 * (double)(grid - wgs) * n / cus;
  return 2.5 + std::max(4.5 + step_us * steps(longest), full) + (n > 1 ? 3.5 + 0.29e-3 * (double)tokens * a.Hq * n : 0.0);
}

// The launches that the other kernels' tiles leave idle, by both models: those kernels take 8 us besides the chain that
// kv_pieces() knows, and have to be behind by a tenth (a fifth for custom masks, a third behind decode rows).  Measured, other
// kernels -> this one, us (8 / 2 heads unless said): prompts of 64 tokens 7.8 -> 7.4, 256 11.4 -> 8.7, 1003 21.9 -> 12.4, 2048
// 34.6 -> 25.8; 1003 tokens on 32 / 8 heads stay (24.8 against 36.9), 500 too (16.6 / 17.4); 128 tokens on a prefix of 4000
// 22.1 -> 18.0, of 16000 27.8 / 27.2; 16 verify steps of 8 tokens on 1000, 8 / 4 heads 32.7 -> 22.9, 32 / 8 heads on 4000
// 99.2 -> 64.8.  60 drawn prefill calls with chunks of up to 4096 tokens: 1.26 times as fast on average.
// Behind decode rows the bound on the lengths may be theirs: then it has to hold for chunks without a prefix too.
// Not with the composition on the device: the grid is that of the bounds, and a workgroup without a tile holds a CU here.
int prefill_packed_pieces(const PrefillArgs& a) {
  const Tuning& tune = tuning();
  const int nseq = a.seq_end - a.seq_begin, forced = tune.prefill_splits;
  if (a.head_dim != 128 || a.G > kCols || tune.prefill_packed == 0 || nseq <= 0 || a.max_q_len <= 0 || a.num_tokens <= 0) return 0;
  if (tune.prefill_packed == 1 && (forced >= 0 || a.max_kv_len <= 0)) return std::max(1, std::min(forced, 64));
  double other = 1e9, spared = 0.0;
  if (tune.prefill_packed != 1) {
    if (a.dist || a.max_kv_len <= 0 || forced > 1 || tune.prefill_staged == 1 || tune.prefill_pipe == 0 || tune.prefill_pipe_nq == 2 ||
        tune.prefill_pipe_tile == 128)
      return 0;
    // (RPA_PREFILL_SPLITS=0: what the model would cut runs whole on the other kernels, nothing else changes)
    if (prefill_unpacked_kv_splits(a, &other) > 1 && forced >= 0) return 0;
    // Masks as words: up to 128 columns of a sequence and kv head always.  103 drawn verify steps of 4 .. 16 tokens on up to 16000: 1.29 .. 3 times
    // as fast as the other kernels with the launch that makes bits, 2.1 x in the geometric mean (by the models 1.65 x): 5 of 4 on 3900 x 32 / 8
    // heads 42.7 -> 20.0 us, 7 of 16 on 2300 x 64 / 8 56.8 -> 24.4, 17 of 8 on 350 x 64 / 8 26.4 -> 20.1, 28 of 16 on 10000 x 32 / 8 415 -> 247.
    // (Up to 2.5 rounds of workgroups: 26 of 16 tokens on 470 x 64 / 8 heads, 3.3 rounds, 33.2 -> 42.0.)
    const int64_t own_tokens = (int64_t)a.num_tokens - a.seq_begin, wgs = own_tokens / (kCols / a.G) * a.Hkv;
    if (a.mask_words && a.max_q_len * a.G <= 4 * kCols && 2 * wgs <= 5 * compute_units()) {
      other = 1e9;
    } else {
      // (a verify step of more than 32 columns whose heads come in fours has the short-chunk tile, which is better than its model: 8 x
      // 16 tokens on 1000, 8 / 2 heads, 23.7 us against 30.1 here, 8 x 8 on 4000, 64 / 8 heads, 91.7 against 60.7.  At 0.6 no one of 64
      // such steps is more than 6 % slower here; up to 12 x 16 on 1000, 32 / 8 heads, 49.2 against 35.8, stay there)
      const bool short_tile = a.max_q_len * a.G > kCols && a.G % 4 == 0;
      const double margin = a.sm.mask_mode == 1 && short_tile ? 0.6 : a.seq_begin > 0 ? 0.65 : a.sm.mask_mode == 1 ? 0.8 : 0.9;
      // (and by a third where this kernel runs more than three rounds: 8 chunks of 35 .. 227 tokens x 64 / 8 heads 56 against 71 us)
      const bool long_grid = wgs > 3 * compute_units();
      other = (long_grid ? std::min(margin, 0.65) : margin) * (8.0 + other);
      // The launch that writes the new tokens is spared: 3 prompts of 47 tokens e4m3 x 8 / 4 heads 11.7 -> 7.9, 2 chunks of 21 on 2661 x 8 / 2 18.2 -> 13.9.
      // Counted in one round of workgroups (6 chunks of 80 on 490 x 40 / 8 19.3, here 24.9), and not for e4m3 pieces (230 tokens on 4277 x 8 / 4 23.0 and 28.1)
      // nor where a tile's rows have an address each (pages of 48: 136 tokens on 3100 x 16 / 8 23.3 and 28.2, 510 on 2894 x 8 / 4 30.0 and 34.5).
      if (a.saves_launch && wgs <= compute_units() && (a.pt.page_size % kTok == 0 || a.pt.page_size == 16)) spared = 3.0;
      if (a.seq_begin > 0 && a.max_q_len < a.max_kv_len) {
        PrefillArgs own = a;
        own.max_kv_len = a.max_q_len;
        double us = 0.0;
        prefill_unpacked_kv_splits(own, &us);
        if (packed_us(own, nseq, 1) >= margin * (8.0 + us)) return 0;
        if (own_tokens * a.Hq > 2ll * compute_units() * kCols) return 0;  // more than two rounds of workgroups
      }
    }
  }
  // (no piece under eight tiles, the partial rows under 256 MB)
  const int64_t row_bytes = (int64_t)a.num_tokens * a.Hq * (kHeadDim + 2) * 4;
  const int64_t cap = forced >= 0 ? 1 : std::min<int64_t>({64, a.max_kv_len / (kWaves * kTok), ((int64_t)256 << 20) / row_bytes});
  int best = 1;
  double best_us = packed_us(a, nseq, 1);
  for (int n : {2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64}) {
    if (n > cap) break;
    const double us = packed_us(a, nseq, n);
    if (us < best_us) {
      best_us = us;
      best = n;
    }
  }
  return best_us < other + (a.fp8 && best > 1 ? 0.0 : spared) ? best : 0;
}

hipError_t launch_prefill_packed(const PrefillArgs& call, int nseq, hipStream_t stream) {
  PrefillArgs a = call;
  const int per = kCols / a.G;
  const int tiles = (a.max_q_len + per - 1) / per;
  const int64_t grid = prefill_grid(a, nseq, tiles, GridShape{per, a.G, 0, false});
  if (grid + a.write_blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  const bool cut = a.kv_splits > 1;
  if (cut && (!a.ws_o || !a.ws_ml || a.kv_splits > 64)) return hipErrorInvalidValue;
  const dim3 g((unsigned)(grid + a.write_blocks), cut ? (unsigned)a.kv_splits : 1u), blk(512);
  const bool cap = a.sm.soft_cap != 0.f || a.sm.round_logits != 0;
  const bool ext = a.sm.xai_len > 0.f || a.sm.mask_mode != 0 || a.sm.q_scale > 0.f;
  const int pg = a.pt.page_size % kTok == 0 ? 1 : a.pt.page_size == 16 ? 2 : 0;
#define RPA_PACKED(P, C, E, ...) hipLaunchKernelGGL((rpa_prefill_packed_kernel<P, C, E, __VA_ARGS__>), g, blk, 0, stream, a, tiles, nseq, per)
#define RPA_PACKED_OPTS(P, F)                            \
  do {                                                   \
    if (a.mask_words) RPA_PACKED(P, false, true, F, true); \
    else if (cap && ext) RPA_PACKED(P, true, true, F);   \
    else if (cap) RPA_PACKED(P, true, false, F);         \
    else if (ext) RPA_PACKED(P, false, true, F);         \
    else RPA_PACKED(P, false, false, F);                 \
  } while (0)
#define RPA_PACKED_PAGES(F)                  \
  do {                                       \
    if (pg == 1) RPA_PACKED_OPTS(1, F);      \
    else if (pg == 2) RPA_PACKED_OPTS(2, F); \
    else RPA_PACKED_OPTS(0, F);              \
  } while (0)
  if (a.fp8) RPA_PACKED_PAGES(true);
  else RPA_PACKED_PAGES(false);
#undef RPA_PACKED_PAGES
#undef RPA_PACKED_OPTS
#undef RPA_PACKED
  return cut ? launch_prefill_combine(a, stream) : hipGetLastError();
}

}  // namespace rpa
