// Split-KV decode for ragged paged attention on gfx950, plus the combine pass,
// the page-table gather and the new-token cache write.
//
// Decode is HBM-bound: every visible KV token is read exactly once.  One
// wavefront owns one (sequence, kv head, kv split) and streams that head's K
// and V rows (adjacent in the head-interleaved cache: K_h | V_h = 2*D elements)
// through the page table with 16-byte loads straight into the MFMA operand
// layout -- no LDS, no barriers, so every wave is independent and the grid is
// just "enough waves to keep ~16 KiB per wave in flight on every SIMD".
//
// Per 32-token block (bf16):
//   S^T[tok, qrow] = K[tok, :] . Q^T        2 x 4 MFMA 16x16x32 (A = K, B = Q^T)
//   online softmax on the 8 scores each lane holds (row stats need one
//   cross-lane max over the 4 lane groups)
//   O^T[dim, qrow] += V^T[dim, tok] . P^T   8 MFMA 16x16x32 (A = V^T, B = P^T)
// The S^T result layout (lane = q row, registers = tokens) is already the B
// operand layout of the second product when the 32 tokens of a block are
// enumerated as slot(g, i) = (i < 4 ? 4g + i : 16 + 4g + i - 4); V is loaded in
// that token order and transposed in registers with v_perm_b32 (two bf16 of
// neighbouring tokens -> one dword), 32 permutes per block.
// GQA: the G query heads of a kv head are the (zero padded) 16 columns of Q^T.

#include <cstdlib>
#include <cstring>
#include <type_traits>

#include "rpa_common.h"
#include "rpa_kernels.h"

// The K / V rows a decode wave streams are read exactly once per launch: non-temporal loads (the `nt` bit: the
// lines are the first to leave the L2 and the memory-side cache again instead of pushing out what is reused).
// C2's decode rows 103.6 -> 90.6 us, C3 360 -> 327 us, C4 238 -> 214 us; -DRPA_DECODE_NT=0 repeats the comparison.
#ifndef RPA_DECODE_NT
#define RPA_DECODE_NT 1
#endif
#if RPA_DECODE_NT
#define RPA_KV_LD16(p) __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p))
#define RPA_KV_LD8(p) __builtin_nontemporal_load(reinterpret_cast<const u32x2_t*>(p))
#else
#define RPA_KV_LD16(p) ld16(p)
#define RPA_KV_LD8(p) ld8(p)
#endif

namespace rpa {

namespace {

constexpr int kBlk = 32;
constexpr int kCacheBits = RPA_DECODE_NT ? 2 : 0;  // of the buffer loads: nt

// What a page holds of a 32-token block, by which the kernels find a block's rows.  kBlocks: whole blocks (a multiple of 32 tokens).
// kHalves: whole halves (a multiple of 16).  Either way a block has one or two page ids, the same in every lane: they
// come as scalars, a row's address is a scalar base and a 32-bit offset.  kLanes: anything else; every lane looks the page of each
// of its ten rows up in LDS and multiplies it out in 64 bits, 0.7 us of arithmetic per block where one wave runs alone.  Pages of 16
// tokens as kLanes and as kHalves: 64 rows of 1000..8000 tokens x 8 heads bf16 254 -> 214 us, e4m3 169 -> 137; 4 rows of
// 1000..4095 25.3 -> 15.4; 5 rows of 64..512 in a bucket 10.2 -> 7.9.  32 rows of 16384 tokens x 8 heads, bf16 / e4m3: 318 / 167 us on
// pages of 64, 319 / 170 on 16 (kHalves), 336 / 231 on 24, 339 / 188 on 4, 337..351 / 204 on 1 (kLanes).
enum Pages { kLanes, kHalves, kBlocks };
constexpr Pages pages_of(int page_size) { return page_size % 32 == 0 ? kBlocks : page_size % 16 == 0 ? kHalves : kLanes; }
struct BlockPages {
  int lo, hi;  // page ids of the block's first and second 16 tokens (kBlocks: lo is both)
};
constexpr int kRowWaves = 8;    // rpa_decode_row_kernel: waves of a workgroup
constexpr int kRowPitch = 132;  // its partial rows in LDS: 128 floats and 16 bytes, so that neighbouring heads' banks differ

__device__ __forceinline__ int tok_slot(int g, int i) {
  return (i < 4) ? (g * 4 + i) : (16 + g * 4 + (i - 4));
}

template <bool FP8>
struct KvRegs;
template <>
struct KvRegs<false> {
  u32x4_t k[2][4];  // [token half][k step]: 8 bf16 of dims 32*s + 8*g ..
  u32x4_t v[8];     // [slot]: 8 bf16 of dims 8*c ..
};
template <>
struct KvRegs<true> {
  u32x4_t k[2][2];  // 32 fp8 of dims 32*g ..
  u32x2_t v[8];     // 8 fp8 of dims 8*c ..
};

struct SeqView {
  const int32_t* pages;  // this sequence's page ids
  int32_t page_size;
  int32_t page_shift;  // >= 0 when page_size is a power of two
  int32_t last_tok;    // kv_len - 1
  // Tokens from fresh_first on are not in the cache yet: they come from the caller's new rows (DecodeArgs.new_k / new_v),
  // fresh_row = row of token fresh_first and this kv head there.  kNoFresh: all are in the cache.
  int32_t fresh_first;
  int32_t fresh_row;
};

constexpr int kNoFresh = 0x7fffffff;

// A wave-uniform condition the optimiser knows nothing else about: without it the rare branches on "this block ends the
// row" are threaded through the whole block's code, which doubles it (8.3 k against 4.5 k instructions).
__device__ __forceinline__ bool rare(bool cond) {
  int v = __builtin_amdgcn_readfirstlane(cond);
  asm("" : "+s"(v));
  return v != 0;
}

__device__ __forceinline__ int page_slot_of(const SeqView& s, int tok) {
  return s.page_shift >= 0 ? (tok >> s.page_shift) : (tok / s.page_size);
}

// Issue the global loads of one 32-token block, whatever it holds.  Token indices are clamped to the last valid token so that
// nothing past kv_len (and nothing past the sequence's page list) is ever dereferenced; clamped rows are masked later.
// kLanes, WINDOW, win / win_first: the LDS window the caller keeps of this row's page ids (entry 0 = page slot win_first);
// without it every lane fetches the ids of its tokens from memory, a dependent round trip in front of the block's loads.
// FRESH: the row's last tokens may come from the caller's new rows instead (SeqView.fresh_first).  Chosen by masks: a lane's
// own branch around the choice costs a drained queue of loads behind it.
// HALF (bf16): heads of 64 dims in rows of 128 whose second half is zero: it is not read.
// PART: the K rows only, the V rows only, or both.
enum BlockPart { kBoth, kOnlyK, kOnlyV };
template <bool FP8, Pages PG, bool WINDOW = false, bool FRESH = false, bool HALF = false, BlockPart PART = kBoth>
__device__ __forceinline__ void load_block(KvRegs<FP8>& r, const DecodeArgs& a, const SeqView& s, const char* kh, const char* vh, int tb, BlockPages page, int c, int g,
                                           const int32_t* win = nullptr, int win_first = 0) {
  const KvAddr& kv = a.kv;
  constexpr int kLaneK = FP8 ? 32 : 16;  // byte offset step of lane group g inside a K row
  constexpr int kLaneV = FP8 ? 8 : 16;   // byte offset step of lane c inside a V row
  // (HALF: the lanes of dims 64.. read those of dims 0.. once more; nothing that they compute is kept)
  const int lane_v = (HALF ? c & 7 : c) * kLaneV;
  int t0[2] = {0, 0};  // first token of each half's page
  if constexpr (PG != kLanes) {
    t0[0] = page_slot_of(s, tb) * s.page_size;
    t0[1] = PG == kHalves ? page_slot_of(s, min(tb + 16, s.last_tok)) * s.page_size : t0[0];
  }
  // (the lane's bytes in the 32-bit offset: a scalar base and one offset per load)
  auto row_of = [&](int tok, int half, const char* cached, const char* fresh, int lane_bytes) __attribute__((always_inline)) -> const char* {
    tok = min(tok, s.last_tok);
    const char* at;
    if constexpr (PG != kLanes) {
      at = cached + (int64_t)(PG == kHalves && half ? page.hi : page.lo) * kv.page_stride + (uint32_t)((tok - t0[half]) * kv.tok_stride + lane_bytes);
    } else {
      const int slot = page_slot_of(s, tok);
      const int pg = WINDOW ? win[slot - win_first] : s.pages[slot];
      at = cached + (int64_t)pg * kv.page_stride + (int64_t)(tok - slot * s.page_size) * kv.tok_stride + lane_bytes;
    }
    if constexpr (FRESH) {
      const char* new_at = fresh + (int64_t)(s.fresh_row + (tok - s.fresh_first) * a.Hkv) * (FP8 || HALF ? 128 : 256) + lane_bytes;
      at += (new_at - at) & -(int64_t)(tok >= s.fresh_first);
    }
    return at;
  };
  if constexpr (PART != kOnlyV) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const char* at = row_of(tb + b * 16 + c, b, kh, a.new_k, g * kLaneK);
#pragma unroll
      for (int st = 0; st < (FP8 || HALF ? 2 : 4); ++st) r.k[b][st] = RPA_KV_LD16(at + st * (FP8 ? 16 : 64));
    }
  }
  if constexpr (PART != kOnlyK) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const char* at = row_of(tb + tok_slot(g, i), i >= 4, vh, a.new_v, lane_v);
      if constexpr (FP8) r.v[i] = RPA_KV_LD8(at);
      else r.v[i] = RPA_KV_LD16(at);
    }
  }
}

// The same of a block whose 32 tokens all lie in the cache.  Buffer loads: a half's first row as the base, one offset per lane
// for all K rows and another for all V rows, what differs between the loads in a scalar: no vector instruction beside the
// loads themselves.  wanted == false: a block that nobody needs, asked for so that the waits behind it count the same on every
// path; its buffers have no bytes, and nothing is fetched.  (kLanes: a block that the piece reads anyway is fetched once more.)
template <bool FP8, Pages PG, bool HALF>
__device__ __forceinline__ void load_full_block(KvRegs<FP8>& r, const DecodeArgs& a, const SeqView& s, const char* kh, const char* vh, int tb, BlockPages page, bool wanted, int c, int g,
                                                const int32_t* win = nullptr, int win_first = 0) {
  if constexpr (PG == kLanes) {
    load_block<FP8, PG, true, false, HALF>(r, a, s, kh, vh, tb, page, c, g, win, win_first);
  } else {
    const KvAddr& kv = a.kv;
    const int off_k = c * kv.tok_stride + g * (FP8 ? 32 : 16);
    const int off_v = 4 * g * kv.tok_stride + (HALF ? c & 7 : c) * (FP8 ? 8 : 16);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int tok = PG == kHalves && h ? tb + 16 : tb;
      const int64_t at = (int64_t)(PG == kHalves && h ? page.hi : page.lo) * kv.page_stride + (int64_t)(tok - page_slot_of(s, tok) * s.page_size) * kv.tok_stride;
      const int behind = PG == kBlocks ? h * 16 * kv.tok_stride : 0, bytes = wanted ? 0x7fffffff : 0;
      const auto k = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kh) + at, 0, bytes, 0x00020000);
      const auto v = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(vh) + at, 0, bytes, 0x00020000);
#pragma unroll
      for (int st = 0; st < (FP8 || HALF ? 2 : 4); ++st)
        r.k[h][st] = __builtin_amdgcn_raw_buffer_load_b128(k, off_k + st * (FP8 ? 16 : 64), behind, kCacheBits);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (FP8) r.v[h * 4 + i] = __builtin_amdgcn_raw_buffer_load_b64(v, off_v, i * kv.tok_stride + behind, kCacheBits);
        else r.v[h * 4 + i] = __builtin_amdgcn_raw_buffer_load_b128(v, off_v, i * kv.tok_stride + behind, kCacheBits);
      }
    }
  }
}

// Any block, out of the cache alone (a new token's slot is read for what stands there): rows past the row's last token are the
// last token's again, by a bound on the lanes' offsets.  (wanted: as above.)
template <bool FP8, Pages PG, bool HALF>
__device__ __forceinline__ void load_cached_block(KvRegs<FP8>& r, const DecodeArgs& a, const SeqView& s, const char* kh, const char* vh, int tb, BlockPages page, bool wanted, int c, int g,
                                                  const int32_t* win, int win_first) {
  if constexpr (PG == kLanes) {
    load_block<FP8, PG, true, false, HALF>(r, a, s, kh, vh, tb, page, c, g, win, win_first);
  } else {
    const KvAddr& kv = a.kv;
    const int lane_k = g * (FP8 ? 32 : 16), lane_v = (HALF ? c & 7 : c) * (FP8 ? 8 : 16);
    const int row_k = c * kv.tok_stride, row_v = 4 * g * kv.tok_stride, bytes = wanted ? 0x7fffffff : 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool hi = PG == kHalves && h && tb + 16 <= s.last_tok;
      const int tok = hi ? tb + 16 : tb, first = PG == kBlocks ? h * 16 : 0;
      const int64_t at = (int64_t)(hi ? page.hi : page.lo) * kv.page_stride + (int64_t)(tok - page_slot_of(s, tok) * s.page_size) * kv.tok_stride;
      const int most = min(s.last_tok - tok, PG == kBlocks ? 31 : 15) * kv.tok_stride;  // offset of the last row that there is
      const auto k = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kh) + at, 0, bytes, 0x00020000);
      const auto v = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(vh) + at, 0, bytes, 0x00020000);
      const int off_k = min(row_k + first * kv.tok_stride, most) + lane_k;
#pragma unroll
      for (int st = 0; st < (FP8 || HALF ? 2 : 4); ++st)
        r.k[h][st] = __builtin_amdgcn_raw_buffer_load_b128(k, off_k + st * (FP8 ? 16 : 64), 0, kCacheBits);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int off_v = min(row_v + (first + i) * kv.tok_stride, most) + lane_v;
        if constexpr (FP8) r.v[h * 4 + i] = __builtin_amdgcn_raw_buffer_load_b64(v, off_v, 0, kCacheBits);
        else r.v[h * 4 + i] = __builtin_amdgcn_raw_buffer_load_b128(v, off_v, 0, kCacheBits);
      }
    }
  }
}

// A row's new token, its last one, in the registers of a block: asked for at the start of the piece that ends the row, put in the
// place of what its cache slot held, and left in that slot.  (No lane's own branch in put(): see load_block.)
template <bool FP8, bool HALF>
struct NewTokenRegs {
  static constexpr int kSteps = FP8 || HALF ? 2 : 4, kStep = FP8 ? 16 : 64, kSrc = FP8 || HALF ? 128 : 256;
  u32x4_t k[kSteps];
  std::conditional_t<FP8, u32x2_t, u32x4_t> v;
  bool on = false;
  __device__ __forceinline__ void load(const DecodeArgs& a, const SeqView& s, int c, int g) {
    const int64_t row = (int64_t)(s.fresh_row + (s.last_tok - s.fresh_first) * a.Hkv) * kSrc;
#pragma unroll
    for (int st = 0; st < kSteps; ++st) k[st] = ld16(a.new_k + row + g * (FP8 ? 32 : 16) + st * kStep);
    const char* vp = a.new_v + row + (HALF ? c & 7 : c) * (FP8 ? 8 : 16);
    if constexpr (FP8) v = ld8(vp);
    else v = ld16(vp);
  }
  __device__ __forceinline__ void put(KvRegs<FP8>& r, int t, int c, int g) const {
    // token t of the block; the rows behind it were its slot's, too, and their values count 0 times something
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int st = 0; st < kSteps; ++st) r.k[b][st] = c + 16 * b >= t ? k[st] : r.k[b][st];
#pragma unroll
    for (int i = 0; i < 8; ++i) r.v[i] = tok_slot(g, i) >= t ? v : r.v[i];
  }
  // kh, vh: this kv head's rows of the cache; page: the id of the token's page, tin: its place there
  __device__ __forceinline__ void store(const KvAddr& kv, const char* kh, const char* vh, int page, int tin, int c, int g) const {
    const int64_t at = (int64_t)page * kv.page_stride + (int64_t)tin * kv.tok_stride;
    char* kp = const_cast<char*>(kh) + at;
    char* vp = const_cast<char*>(vh) + at;
    const u32x4_t zero = {0u, 0u, 0u, 0u};
    if (c == 0) {
#pragma unroll
      for (int st = 0; st < kSteps; ++st) st16(kp + g * (FP8 ? 32 : 16) + st * kStep, k[st]);
      if constexpr (HALF) {
        st16(kp + g * 16 + 128, zero);
        st16(kp + g * 16 + 192, zero);
      }
    }
    if (g == 0) {
      if constexpr (FP8) *reinterpret_cast<u32x2_t*>(vp + c * 8) = v;
      else st16(vp + c * 16, HALF && c >= 8 ? zero : v);
    }
  }
};

// A row's new token, its last one, on its way into the cache: the wave whose piece ends the row copies the K and V rows of its
// kv head, 16 bytes per lane.  It is asked for in front of the piece's blocks and stored behind them.  (Nobody reads the slot
// meanwhile: the blocks take new tokens from the caller's rows.  Taken out of the registers of the row's last block instead, it
// was a dozen branches in the block loop, each lane its own way; see load_block.)
template <bool FP8, bool HALF>
struct NewToken {
  static constexpr int kRow = FP8 ? 128 : 256, kSrc = HALF ? 128 : kRow;  // bytes of a row in the cache, in the caller's keys / values
  u32x4_t data = {0u, 0u, 0u, 0u};
  bool on = false;
  __device__ __forceinline__ void load(const DecodeArgs& a, const SeqView& s, int lane) {
    const int at = (lane & 15) * 16;
    if (lane < 32 && at < kSrc)
      data = ld16((lane < 16 ? a.new_k : a.new_v) + (int64_t)(s.fresh_row + (s.last_tok - s.fresh_first) * a.Hkv) * kSrc + at);
  }
  // kh, vh: this kv head's rows of the cache; page: the id of the token's page, tin: its place there
  __device__ __forceinline__ void store(const KvAddr& kv, const char* kh, const char* vh, int page, int tin, int lane) const {
    const int at = (lane & 15) * 16;
    if (lane < 32 && at < kRow)
      st16(const_cast<char*>(lane < 16 ? kh : vh) + (int64_t)page * kv.page_stride + (int64_t)tin * kv.tok_stride + at, data);
  }
};

// The general path of a block's scores: soft cap (if any), temperature, the logit rounded (if asked), in log2 units.
// The constants are folded once per row, cap tanh(s scale / cap) temp log2e = k2 - 2 k2 / (2^(s k1) + 1), and a choice
// that is the same for the whole call is asked once per block: asked per score, as it was first, each score's chain of
// v_exp_f32 and v_rcp_f32 ran alone between two branches, with one wave per SIMD to wait for it.
// 32 rows of 8000..16000 tokens, soft cap, 8 kv heads: e4m3 158 -> 140 us, on 256-wide heads 350.6 -> 299.6.
// The bf16 kernels have no register to spare beside the blocks in flight: the constants stand in scalar registers.
// LOOPS, a loop for either rounding, is for the balanced kernels on whole pages: rounded e4m3 logits are the faster for it (rows as
// above, rounded to bf16 with the cap 149 -> 136 us, without 150 -> 140), everything else is level.  On other pages e4m3 loses by it
// (capped rows as above on 16-token pages 138 -> 143 us, on 24-token pages 210 -> 213).
struct LogitOpts {
  float k1, k2;
  bool capped;
  int round_mode;  // 1 = bf16, 2 = f16
  __device__ __forceinline__ static float scalar(float x) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x))); }
  __device__ __forceinline__ void set(const SoftmaxOpts& sm, float scale, float temp) {
    capped = sm.soft_cap != 0.f;
    round_mode = sm.round_logits;
    k1 = scalar(capped ? scale * (1.0f / sm.soft_cap) * (2.0f * kLog2e) : 0.f);
    k2 = scalar((capped ? sm.soft_cap : scale) * temp * (round_mode ? 1.0f : kLog2e));
  }
  template <bool LOOPS = false>
  __device__ __forceinline__ void apply(float (&x)[8]) const {
    if (capped) {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = __builtin_fmaf(__builtin_amdgcn_rcpf(fast_exp2(x[i] * k1) + 1.0f), -2.0f * k2, k2);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = x[i] * k2;
    }
    if constexpr (LOOPS) {
      if (round_mode == 1) {
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = bf16_round(x[i]) * kLog2e;
      } else if (round_mode) {
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = f16_round(x[i]) * kLog2e;
      }
    } else if (round_mode) {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = round_logit(x[i], round_mode) * kLog2e;
    }
  }
};

struct ScoreOpts {
  float scale2;       // sm_scale * k_scale * temperature * log2(e)  (plain path)
  LogitOpts general;  // soft cap and rounding                       (general path)
  float mask2;      // mask value in log2 units (finite)
  int t_lo;         // first visible token (sliding window), 0 otherwise
  int kv_len;
};

// K operands (A of S^T = K Q^T) of one 32-token block: [token half][k step]
template <bool FP8, bool HALF = false>
__device__ __forceinline__ void k_operands(const KvRegs<FP8>& r, u32x4_t (&kA)[2][4]) {
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    if constexpr (FP8) {
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const uint32_t w0 = r.k[b][st >> 1][(st & 1) * 2 + 0];
        const uint32_t w1 = r.k[b][st >> 1][(st & 1) * 2 + 1];
        const u32x2_t lo = fp8x4_to_bf16x4(w0);
        const u32x2_t hi = fp8x4_to_bf16x4(w1);
        kA[b][st] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
      }
    } else {
#pragma unroll
      for (int st = 0; st < (HALF ? 2 : 4); ++st) kA[b][st] = r.k[b][st];
    }
  }
}

// V^T operands (A of O^T = V^T P^T), one per output dim j of the lane's 8-dim chunk
template <bool FP8>
__device__ __forceinline__ void v_operands(const KvRegs<FP8>& r, u32x4_t (&vA)[8]) {
  if constexpr (FP8) {
    // r.v[i] = 8 fp8 (dims 8c .. 8c+7) of token slot i.  A byte permute first pairs the bytes of
    // two neighbouring tokens for two dims (t0 d, t1 d, t0 d+1, t1 d+1), then each half converts
    // straight to a bf16 pair: 3 instructions per 4 values.
#pragma unroll
    for (int tp = 0; tp < 4; ++tp)
#pragma unroll
      for (int dp = 0; dp < 4; ++dp) {
        const uint32_t lo_tok = r.v[2 * tp][dp >> 1], hi_tok = r.v[2 * tp + 1][dp >> 1];
        // selector bytes: 0-3 pick from lo_tok (second operand), 4-7 from hi_tok (first operand)
        const uint32_t sel = (dp & 1) ? 0x07030602u : 0x05010400u;
        const uint32_t mixed = __builtin_amdgcn_perm(hi_tok, lo_tok, sel);
        vA[2 * dp][tp] = fp8x2_to_bf16x2(mixed, false);
        vA[2 * dp + 1][tp] = fp8x2_to_bf16x2(mixed, true);
      }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
      const int jj = j >> 1;
      vA[j] = u32x4_t{__builtin_amdgcn_perm(r.v[1][jj], r.v[0][jj], sel),
                      __builtin_amdgcn_perm(r.v[3][jj], r.v[2][jj], sel),
                      __builtin_amdgcn_perm(r.v[5][jj], r.v[4][jj], sel),
                      __builtin_amdgcn_perm(r.v[7][jj], r.v[6][jj], sel)};
    }
  }
}

__device__ __forceinline__ float max8(const float (&x)[8]) {
  return fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
}

struct Nothing {
  __device__ __forceinline__ void operator()() const {}
};

// `taken` runs when the block's registers have been read (FP8: its operands are in registers of their own): the place to ask for
// another block in the same registers.
template <int MT, bool FP8, bool CAP, bool HALF = false, bool LOOPS = false, class Taken = Nothing>
__device__ __forceinline__ void compute_block(const KvRegs<FP8>& r, const u32x4_t (&qB)[MT][4],
                                              f32x4_t (&acc)[MT][8], float (&m)[MT], float (&l)[MT],
                                              const ScoreOpts& so, int tb, int g, const Taken& taken = Taken()) {
  constexpr bool kEarly = !std::is_same_v<Taken, Nothing>;
  u32x4_t kA[2][4];
  k_operands<FP8, HALF>(r, kA);
  f32x4_t s_of[kEarly ? MT : 1][2];
  auto scores = [&](int mt, f32x4_t (&s)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      s[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int st = 0; st < (HALF ? 2 : 4); ++st) s[b] = mfma16(kA[b][st], qB[mt][st], s[b]);
    }
  };
  if constexpr (kEarly) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) scores(mt, s_of[mt]);
  }
  u32x4_t vA[8];
  v_operands<FP8>(r, vA);
  if constexpr (kEarly) {
#pragma unroll
    for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(vA[j]));  // made here, not where they are used
    taken();
  }
  const bool need_mask = (tb + kBlk > so.kv_len) || (tb < so.t_lo);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    f32x4_t(&s)[2] = s_of[kEarly ? mt : 0];
    if constexpr (!kEarly) scores(mt, s);
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = CAP ? s[i >> 2][i & 3] : s[i >> 2][i & 3] * so.scale2;
    if constexpr (CAP) so.general.apply<LOOPS>(x);
    // (the maximum of unmasked scores in front of the branch: behind it every one of them would be canonicalised first)
    float mx = max8(x);
    if (need_mask) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int tok = tb + tok_slot(g, i);
        if (tok >= so.kv_len || tok < so.t_lo) x[i] = so.mask2;
      }
      mx = max8(x);
    }
    mx = swap_max(swap16_max(mx));
    const float m_new = fmaxf(m[mt], mx);
    const float alpha = fast_exp2(m[mt] - m_new);
    float p[8];
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      p[i] = fast_exp2(x[i] - m_new);
      ps += p[i];
    }
    l[mt] = l[mt] * alpha + ps;
    m[mt] = m_new;
    const u32x4_t pB = u32x4_t{pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3]),
                               pack_bf16x2(p[4], p[5]), pack_bf16x2(p[6], p[7])};
    if constexpr (FP8) {
      // fp8 blocks are VALU-bound (dequantisation): skip the accumulator rescale unless the
      // running max moved in some lane, which is rare after the first blocks
      if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[mt][j] = acc[mt][j] * alpha;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[mt][j] = mfma16(vA[j], pB, acc[mt][j]);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        acc[mt][j] = acc[mt][j] * alpha;
        acc[mt][j] = mfma16(vA[j], pB, acc[mt][j]);
      }
    }
  }
}

__device__ __forceinline__ int first_block_token(int kv_len, int window) {
  const int t_lo = (window > 0) ? max(0, kv_len - window) : 0;
  return t_lo & ~(kBlk - 1);
}

// Where a wave leaves the result of one piece of work: the finished bf16 rows in `out`, or
// unnormalised partial rows plus (max, sum) in the workspace, slot `base` + query head
// (fixed split plan) or `base` + row inside the group of 16 (balanced plan).
struct PartDest {
  bool final_rows;
  bool by_head;
  int64_t base;
};

// Q^T operands of one (query token, kv head, group of 16 query heads): column c = query head
// row0 + 16*mt + c of the kv head, zero beyond the G real ones.
template <int MT, bool FP8>
__device__ __forceinline__ void load_queries(const DecodeArgs& a, int tq, int hk, int row0, int c, int g,
                                             u32x4_t (&qB)[MT][4]) {
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int row = row0 + mt * 16 + c;
    const uint16_t* qp = a.q + ((int64_t)tq * a.Hq + (int64_t)hk * a.G + row) * a.q_dim;
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const int d0 = FP8 ? g * 32 + st * 8 : st * 32 + g * 8;
      qB[mt][st] = ld_query(qp, row < a.G ? d0 : a.q_dim, a.q_dim);
    }
  }
}

template <int MT, bool FP8>
__device__ __forceinline__ void requantise_queries(const DecodeArgs& a, u32x4_t (&qB)[MT][4]) {
  if (a.sm.q_scale > 0.f) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int st = 0; st < 4; ++st) qB[mt][st] = requantise_q(qB[mt][st], a.sm.q_scale, FP8);
  }
}

// Leave the result of one piece of work: lane (c, g) holds q row c, dims 32g + 8r + j in
// acc[mt][j][r].
template <int MT, bool THROUGH = false>
__device__ __forceinline__ void write_rows(const DecodeArgs& a, const f32x4_t (&acc)[MT][8], const float (&m)[MT],
                                           const float (&l)[MT], int tq, int hk, int row0, const PartDest dest,
                                           float vs, int c, int g) {
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    float lt = l[mt];
    lt += __shfl_xor(lt, 16);
    lt += __shfl_xor(lt, 32);
    const int row = row0 + mt * 16 + c;
    if (row >= a.G) continue;
    const int head = hk * a.G + row;
    if (dest.final_rows) {
      const float inv = a.sm.sink ? vs * sink_inverse(m[mt], lt, sink_logit(a.sm.sink, a.sm.round_logits, head)) : vs / lt;
      uint16_t* op = a.out + ((int64_t)tq * a.Hq + head) * a.q_dim + g * 32;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (g * 32 + r * 8 >= a.q_dim) break;
        u32x4_t w;
#pragma unroll
        for (int jp = 0; jp < 4; ++jp)
          w[jp] = pack_bf16x2(acc[mt][2 * jp][r] * inv, acc[mt][2 * jp + 1][r] * inv);
        st16(op + r * 8, w);
      }
    } else {
      const int64_t slot = dest.base + (dest.by_head ? head : row - row0);
      float* wo = a.ws_o + slot * 128 + g * 32;
      // merged inside the same launch: the rows are written through to device scope, so that the
      // merging wave (on another part of the GPU, behind another L2) reads them without any
      // cache-wide write-back or invalidate
      constexpr bool through = THROUGH;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        f32x4_t w0 = {acc[mt][0][r] * vs, acc[mt][1][r] * vs, acc[mt][2][r] * vs, acc[mt][3][r] * vs};
        f32x4_t w1 = {acc[mt][4][r] * vs, acc[mt][5][r] * vs, acc[mt][6][r] * vs, acc[mt][7][r] * vs};
        if (through) {
          // s_nop: a store of more than 8 bytes needs a wait state in front of a vector instruction that overwrites its data.  The
          // compiler sees to that behind its own stores, not behind these: in one build the next row's address went straight into
          // the registers of a store (bf16, whole pages, soft cap), and 3 of 2250 random batches came out wrong.
          asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 0" ::"v"(wo + r * 8), "v"(w0) : "memory");
          asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 0" ::"v"(wo + r * 8 + 4), "v"(w1) : "memory");
        } else {
          *reinterpret_cast<f32x4_t*>(wo + r * 8) = w0;
          *reinterpret_cast<f32x4_t*>(wo + r * 8 + 4) = w1;
        }
      }
      if (g == 0) {
        if (through) {
          __hip_atomic_store(a.ws_ml + slot * 2 + 0, m[mt], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(a.ws_ml + slot * 2 + 1, lt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
          a.ws_ml[slot * 2 + 0] = m[mt];
          a.ws_ml[slot * 2 + 1] = lt;
        }
      }
    }
  }
}

// One row: query token tq of sequence seq, which sees kv_len tokens; new tokens start at position fresh_first, whose
// query token is fresh_tq; its page ids start at page_indices[page0].
struct RowRef {
  int seq, tq, kv_len, fresh_first, fresh_tq;
  int64_t page0;
};

__device__ __forceinline__ int owner_of_token(const int32_t* cu_q_lens, int num_seqs, int tok) {
  int lo = 0, hi = num_seqs;  // last i with cu_q_lens[i] <= tok (zero-length sequences are skipped)
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cu_q_lens[mid] <= tok) lo = mid; else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ int64_t first_page(const DecodeArgs& a, int seq, int cu_kv) {
  if (!a.pt.cu_kv_lens) return (int64_t)seq * a.pt.pages_per_seq;
  const int P = a.pt.page_size;
  return (P & (P - 1)) == 0 ? cu_kv >> (31 - __builtin_clz(P)) : cu_kv / P;
}

// Row `index` of the fixed plan: decode row `index`, or (token_rows) query token `index` of whatever sequence owns it.
// false: nothing there.
// Everything that the batch holds about the row is asked for at once.  With each answer asking the next question (composition, owner by a
// binary search, lengths, page offset) it was 1.9 us of a launch of 8, for a bucket of 5 rows.
__device__ __forceinline__ bool fixed_row(const DecodeArgs& a, int index, RowRef& row) {
  const int32_t* cu_kv_lens = a.pt.cu_kv_lens ? a.pt.cu_kv_lens : a.pt.kv_lens;  // (any words that are there)
  if (a.token_rows) {
    int cu_kv;
    if (a.num_seqs < 64) {  // a sequence per lane
      const int lane = threadIdx.x & 63, own = min(lane, a.num_seqs - 1);
      const int seqs_now = scalar_load_i32(a.dist ? a.dist + 2 : a.pt.kv_lens);
      const int q0 = a.pt.cu_q_lens[min(lane, a.num_seqs)], kv = a.pt.kv_lens[own], at = cu_kv_lens[own];
      const int seqs = a.dist ? max(min(a.num_seqs, seqs_now), 0) : a.num_seqs;
      if (index >= __builtin_amdgcn_readlane(q0, seqs)) return false;
      row.tq = index;
      row.seq = max(__builtin_popcountll(__builtin_amdgcn_ballot_w64(lane < seqs && q0 <= index)) - 1, 0);
      row.fresh_tq = __builtin_amdgcn_readlane(q0, row.seq);
      row.fresh_first = __builtin_amdgcn_readlane(kv, row.seq) - (__builtin_amdgcn_readlane(q0, row.seq + 1) - row.fresh_tq);
      cu_kv = __builtin_amdgcn_readlane(at, row.seq);
    } else {
      const int seqs = a.dist ? min(a.num_seqs, scalar_load_i32(a.dist + 2)) : a.num_seqs;
      if (index >= scalar_load_i32(a.pt.cu_q_lens + seqs)) return false;
      row.tq = index;
      row.seq = __builtin_amdgcn_readfirstlane(owner_of_token(a.pt.cu_q_lens, seqs, index));
      row.fresh_tq = scalar_load_i32(a.pt.cu_q_lens + row.seq);
      row.fresh_first = scalar_load_i32(a.pt.kv_lens + row.seq) - (scalar_load_i32(a.pt.cu_q_lens + row.seq + 1) - row.fresh_tq);
      cu_kv = scalar_load_i32(cu_kv_lens + row.seq);
    }
    row.kv_len = row.fresh_first + (index - row.fresh_tq) + 1;
    row.page0 = first_page(a, row.seq, cu_kv);
    return row.fresh_first >= 0;
  }
  // (static-shape mode: the number of decode rows comes from the device; the grid's rows are all sequences of the call)
  const int rows_now = scalar_load_i32(a.dist ? a.dist : a.pt.kv_lens);
  row.seq = index;
  row.kv_len = scalar_load_i32(a.pt.kv_lens + index);
  row.tq = row.fresh_tq = scalar_load_i32(a.pt.cu_q_lens + index);
  const int cu_kv = scalar_load_i32(cu_kv_lens + index);
  if (index >= (a.dist ? min(a.num_rows, rows_now) : a.num_rows)) return false;
  row.fresh_first = row.kv_len - 1;
  row.page0 = first_page(a, index, cu_kv);
  return row.kv_len > 0;
}

// One wave, one (row, kv head, group of 16 query heads), tokens [t_begin, t_end): unnormalised output rows, maxima, sums.
template <int MT, bool FP8, Pages PG, bool CAP, bool HALF, int WAVES>
__device__ __forceinline__ void decode_segment(const DecodeArgs& a, const RowRef& row, int hk, int rg, int t_lo,
                                               int t_begin, int t_end, f32x4_t (&acc)[MT][8], float (&m)[MT], float (&l)[MT],
                                               int lane) {
  const int kv_len = row.kv_len;
  const int c = lane & 15, g = lane >> 4;
  const int nblk = (t_end - t_begin + kBlk - 1) / kBlk;

  SeqView sv;
  sv.page_size = a.pt.page_size;
  sv.page_shift = ((sv.page_size & (sv.page_size - 1)) == 0) ? (31 - __builtin_clz(sv.page_size)) : -1;
  sv.last_tok = kv_len - 1;
  // Sequence metadata and page ids go through the scalar cache: nothing writes them while the
  // kernel runs, and a scalar load is not counted by vmcnt, so waiting for a page id never
  // drains the block prefetch issued just before it.
  sv.pages = a.pt.page_indices + row.page0;

  const char* kh = a.kv.k_base + (int64_t)hk * a.kv.head_stride;
  const char* vh = a.kv.v_base + (int64_t)hk * a.kv.head_stride;
  sv.fresh_first = a.new_k ? row.fresh_first : kNoFresh;
  sv.fresh_row = row.fresh_tq * a.Hkv + hk;

  // ---- software pipeline: two blocks are in flight or in use.  The piece's last block goes first: it may end the row, or reach
  // into its new tokens, and takes an address per lane and row; the blocks behind it are full ones of the cache, so the
  // loop has one kind of loads, stands once in the code for it, and its waits stay counted: with a choice of loads in the
  // loop the compiler closes it with a block that has a way past them and drains the queue in front of every use.  A piece of two
  // blocks asks for those two and no more.  16 rows of 32 k tokens x 8 heads 316 -> 304 us (7.06 TB/s), 8 rows of 64..512 on
  // pages of 64 8.4 -> 7.2.
  const int full = nblk - 1;  // blocks but the last
  const int t_last = t_begin + full * kBlk;
  auto page_of = [&](int tb) -> BlockPages {
    BlockPages p = {};
    if constexpr (PG != kLanes) p.lo = scalar_load_i32(sv.pages + __builtin_amdgcn_readfirstlane(page_slot_of(sv, tb)));
    if constexpr (PG == kHalves) p.hi = scalar_load_i32(sv.pages + __builtin_amdgcn_readfirstlane(page_slot_of(sv, min(tb + 16, sv.last_tok))));
    return p;
  };
  // (a chunk's query tokens as rows: its new tokens may reach over several blocks, a few at most)
  int first = 0;
  if (a.token_rows)
    while (full - first > 0 && t_last - first * kBlk > sv.fresh_first) ++first;
  const int n = full - first;  // full blocks of the cache
  auto next_tok = [&](int b) { return t_begin + min(b, max(n - 1, 0)) * kBlk; };
  const BlockPages pg_last = page_of(t_last);
  BlockPages pg_next = page_of(next_tok(0));
  NewToken<FP8, HALF> fresh;
  fresh.on = a.new_k && t_end == kv_len;
  if (fresh.on) fresh.load(a, sv, lane);

  // ---- Q^T operands: column c = query head (row0 + 16*mt + c) of this kv head ----
  const int tq = row.tq;
  const int row0 = rg * 16 * MT;
  u32x4_t qB[MT][4];
  load_queries<MT, FP8>(a, tq, hk, row0, c, g, qB);
  requantise_queries<MT, FP8>(a, qB);

  ScoreOpts so;
  const float ks = a.k_scale ? scalar_load_f32(a.k_scale + hk) : 1.0f;
  // the one query of a decode row sits at position kv_len - 1
  const float temp = xai_factor(kv_len - 1, a.sm.xai_len);
  const float scale = a.sm.sm_scale * ks * (a.sm.q_scale > 0.f ? a.sm.q_scale : 1.0f);
  so.scale2 = scale * kLog2e * temp;
  so.general.set(a.sm, scale, temp);
  so.mask2 = fmaxf(a.sm.mask_value * kLog2e, -3.0e38f);
  so.t_lo = t_lo;
  so.kv_len = kv_len;

#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    m[mt] = -INFINITY;
    l[mt] = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[mt][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  // Pages smaller than half a block: the ids of the next kWinSmallPages pages wait in the wave's LDS window and
  // every lane looks its token rows up there; fetched from memory per block they were a dependent round
  // trip in front of every block's loads, behind which the loads already in flight had to drain (page size
  // 16: 2.6 TB/s where pages of 64 stream 5.8).  The window moves on every kWinSmallPages pages, at the
  // price of one drained queue.
  __shared__ int32_t seg_windows[PG != kLanes ? 1 : WAVES][PG != kLanes ? 1 : kWinSmallPages];  // [wave][entry]
  const int32_t* win = nullptr;
  int win_first = 0;
  auto cover = [&](int tb) __attribute__((always_inline)) {  // make the window hold the pages of block tb
    if constexpr (PG == kLanes) {
      const int lo = page_slot_of(sv, tb), hi = page_slot_of(sv, min(tb + kBlk - 1, sv.last_tok));
      if (!win || lo < win_first || hi - win_first >= kWinSmallPages) {
        int32_t* mine = seg_windows[__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)];
        // (from the piece's first page if the whole piece fits)
        const int begin = page_slot_of(sv, t_begin);
        win_first = __builtin_amdgcn_readfirstlane(page_slot_of(sv, t_end - 1) - begin < kWinSmallPages ? begin : lo);
        copy_page_window<kWinSmallPages>(sv.pages, page_slot_of(sv, sv.last_tok), mine, win_first, lane);
        wait_all_loads();
        win = mine;
      }
    }
  };
  KvRegs<FP8> ra, rb;
  for (int b = 1; b <= first; ++b) {
    const int tb = t_last - b * kBlk;
    cover(tb);
    load_block<FP8, PG, PG == kLanes, true, HALF>(rb, a, sv, kh, vh, tb, page_of(tb), c, g, win, win_first);
    compute_block<MT, FP8, CAP, HALF>(rb, qB, acc, m, l, so, tb, g);
  }
  cover(t_last);
  load_block<FP8, PG, PG == kLanes, true, HALF>(ra, a, sv, kh, vh, t_last, pg_last, c, g, win, win_first);
  int in_a = t_last;  // first tokens of the blocks in ra, rb
  int asked = 1;      // full blocks asked for; beyond n they are the last one again and not wanted
  cover(next_tok(0));
  load_full_block<FP8, PG, HALF>(rb, a, sv, kh, vh, next_tok(0), pg_next, n > 0, c, g, win, win_first);
  while (asked < n) {
    pg_next = page_of(next_tok(asked));
    compute_block<MT, FP8, CAP, HALF>(ra, qB, acc, m, l, so, in_a, g);
    cover(next_tok(asked));
    load_full_block<FP8, PG, HALF>(ra, a, sv, kh, vh, next_tok(asked), pg_next, true, c, g, win, win_first);
    in_a = next_tok(asked);
    pg_next = page_of(next_tok(asked + 1));
    compute_block<MT, FP8, CAP, HALF>(rb, qB, acc, m, l, so, next_tok(asked - 1), g);
    cover(next_tok(asked + 1));
    load_full_block<FP8, PG, HALF>(rb, a, sv, kh, vh, next_tok(asked + 1), pg_next, asked + 1 < n, c, g, win, win_first);
    asked += 2;
  }
  compute_block<MT, FP8, CAP, HALF>(ra, qB, acc, m, l, so, in_a, g);
  if (asked == n) compute_block<MT, FP8, CAP, HALF>(rb, qB, acc, m, l, so, next_tok(n - 1), g);
  if (fresh.on) {
    const int slot = __builtin_amdgcn_readfirstlane(page_slot_of(sv, sv.last_tok));
    fresh.store(a.kv, kh, vh, scalar_load_i32(sv.pages + slot), sv.last_tok - slot * sv.page_size, lane);
  }
}

// ---- fixed split plan: grid = (max_splits * rows, 1, head groups * row groups), splits fastest (rows do
// not sit on a grid dimension of their own: that one ends at 65535); block = NW waves
template <int MT, bool FP8, Pages PG, bool CAP, bool HALF = false>
__global__ __launch_bounds__(256, 2) void rpa_decode_splitkv_kernel(const DecodeArgs a) {
  const int nsp = max(a.max_splits, 1);
  const int index = (int)(blockIdx.x / (unsigned)nsp);
  const int split = (int)blockIdx.x - index * nsp;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = blockDim.x >> 6;
  const int head_groups = (a.Hkv + nw - 1) / nw;
  const int hg = blockIdx.z % head_groups;
  const int rg = blockIdx.z / head_groups;
  const int hk = hg * nw + wave;
  RowRef row;
  if (hk >= a.Hkv || !fixed_row(a, index, row)) return;

  const int t_lo = (a.sm.window > 0) ? max(0, row.kv_len - a.sm.window) : 0;
  const int t0 = t_lo & ~(kBlk - 1);
  const int t_begin = t0 + split * a.chunk;
  if (t_begin >= row.kv_len) return;
  // the last split runs to kv_len even if the host's length bound was too small
  const int t_end = (split == a.max_splits - 1) ? row.kv_len : min(row.kv_len, t_begin + a.chunk);
  PartDest dest;
  dest.final_rows = a.max_splits == 1;
  dest.by_head = true;
  dest.base = ((int64_t)index * a.max_splits + split) * a.Hq;
  f32x4_t acc[MT][8];
  float m[MT], l[MT];
  const float vs = a.v_scale ? scalar_load_f32(a.v_scale + hk) : 1.0f;
  decode_segment<MT, FP8, PG, CAP, HALF, 4>(a, row, hk, rg, t_lo, t_begin, t_end, acc, m, l, lane);
  write_rows<MT>(a, acc, m, l, row.tq, hk, rg * 16 * MT, dest, vs, lane & 15, lane >> 4);
}

// ---- rows by workgroups: grid = (pieces * rows, 1, kv heads * row groups); one workgroup of kRowWaves waves deals the blocks of a
// row, or of one of max_splits pieces of it, out among them and merges their partial rows in LDS: two barriers and 8 KB per 2 query
// heads.  8 waves: the registers allow two per SIMD.  Whole short rows are bound by latency (the split kernel and its merge are
// two launches; a few rows of up to 255 tokens 10.2 -> 7.5 us), pieces that fill the chip by what a CU draws:
// 32 rows of 800..1000 tokens x 8 heads, whole, 31.5 -> 24.1 us.  Which rows come here: row_plan().
template <bool FP8, Pages PG, bool CAP, bool HALF = false>
__global__ __launch_bounds__(kRowWaves * 64, 2) void rpa_decode_row_kernel(const DecodeArgs a) {
  extern __shared__ float row_parts[];  // [wave][query head of the group][kRowPitch]
  __shared__ float row_ml[kRowWaves][16][2];
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hk = (int)blockIdx.z % a.Hkv, rg = (int)blockIdx.z / a.Hkv;
  const int nsp = max(a.max_splits, 1), index = (int)(blockIdx.x / (unsigned)nsp), split = (int)blockIdx.x - index * nsp;
  RowRef row;
  if (!fixed_row(a, index, row)) return;
  const int t_lo = (a.sm.window > 0) ? max(0, row.kv_len - a.sm.window) : 0;
  const int t0 = (t_lo & ~(kBlk - 1)) + split * a.chunk;
  // (the last split runs to kv_len even if the host's length bound was too small)
  const int t1 = split == nsp - 1 ? row.kv_len : min(row.kv_len, t0 + a.chunk);
  if (t0 >= t1) return;
  const int piece = ((t1 - t0 + kBlk - 1) / kBlk + kRowWaves - 1) / kRowWaves * kBlk;
  const int used = (t1 - t0 + piece - 1) / piece;  // waves with work
  const int heads = min(16, a.G - rg * 16);
  const float vs = a.v_scale ? scalar_load_f32(a.v_scale + hk) : 1.0f;
  f32x4_t acc[1][8];
  float m[1], l[1];
  if (wave < used) {
    const int t_begin = t0 + wave * piece;
    decode_segment<1, FP8, PG, CAP, HALF, kRowWaves>(a, row, hk, rg, t_lo, t_begin, min(t1, t_begin + piece),
                                                               acc, m, l, lane);
    float lt = l[0];
    lt += __shfl_xor(lt, 16);
    lt += __shfl_xor(lt, 32);
    if (g == 0) {
      row_ml[wave][c][0] = m[0];
      row_ml[wave][c][1] = lt;
    }
  }
  __syncthreads();
  if (wave < used && c < heads) {
    float top = row_ml[0][c][0];
    for (int w = 1; w < used; ++w) top = fmaxf(top, row_ml[w][c][0]);
    const float share = fast_exp2(m[0] - top);
    float* to = row_parts + (wave * heads + c) * kRowPitch + g * 32;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      *reinterpret_cast<f32x4_t*>(to + r * 8) =
          f32x4_t{acc[0][0][r], acc[0][1][r], acc[0][2][r], acc[0][3][r]} * share;
      *reinterpret_cast<f32x4_t*>(to + r * 8 + 4) =
          f32x4_t{acc[0][4][r], acc[0][5][r], acc[0][6][r], acc[0][7][r]} * share;
    }
  }
  __syncthreads();
  for (int at = (int)threadIdx.x; at < heads * 64; at += kRowWaves * 64) {
    const int h = at >> 6, d = (at & 63) * 2;  // two dims of one query head
    const int head = hk * a.G + rg * 16 + h;
    float top = row_ml[0][h][0];
    for (int w = 1; w < used; ++w) top = fmaxf(top, row_ml[w][h][0]);
    float den = 0.f, x = 0.f, y = 0.f;
    for (int w = 0; w < used; ++w) {
      den += row_ml[w][h][1] * fast_exp2(row_ml[w][h][0] - top);
      const float* from = row_parts + (w * heads + h) * kRowPitch + d;
      x += from[0];
      y += from[1];
    }
    if (nsp > 1) {
      const int64_t slot = ((int64_t)index * nsp + split) * a.Hq + head;
      *reinterpret_cast<f32x2_t*>(a.ws_o + slot * 128 + d) = f32x2_t{x * vs, y * vs};
      if (d == 0) *reinterpret_cast<f32x2_t*>(a.ws_ml + slot * 2) = f32x2_t{top, den};
      continue;
    }
    const float inv = a.sm.sink ? vs * sink_inverse(top, den, sink_logit(a.sm.sink, a.sm.round_logits, head)) : vs / den;
    if (d < a.q_dim)
      *reinterpret_cast<uint32_t*>(a.out + ((int64_t)row.tq * a.Hq + head) * a.q_dim + d) = pack_bf16x2(x * inv, y * inv);
  }
}

// ---- balanced plan ------------------------------------------------------------------------
// All 32-token blocks of the batch are laid out in one line -- sequence by sequence, inside a
// sequence unit by unit, inside a unit block by block -- and workgroup j takes blocks
// [j * pw, (j + 1) * pw): every workgroup streams the same number of KV bytes whatever the
// ragged lengths are, and nothing about the lengths has to be known on the host.  A unit is a
// group of NW neighbouring kv heads (x a group of 16 query heads): the NW waves of a workgroup
// walk the same tokens of neighbouring heads, whose rows are adjacent in the head-interleaved
// cache.  A workgroup crosses at most a few unit borders; units it covers completely are
// finished in place, the cut ones (at most its first and its last) leave partial rows in the
// workspace slots 2w and 2w + 1 of its waves w.
__device__ __forceinline__ int seq_blocks(int kv_len, int window) {
  return kv_len > 0 ? (kv_len - first_block_token(kv_len, window) + kBlk - 1) / kBlk : 0;
}

__device__ __forceinline__ int wave_inclusive_scan(int v, int lane) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int n = __shfl_up(v, off);
    if (lane >= off) v += n;
  }
  return v;
}

// Linear block indices are 32-bit: a batch holds fewer than 2^31 (32-token block, unit) pairs.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// total number of blocks of sequences [0, upto) -- all lanes of the wave must call it
__device__ __forceinline__ int blocks_before(const DecodeArgs& a, int upto, int lane) {
  int total = 0;
  for (int s0 = 0; s0 < upto; s0 += 64) {
    const int s = s0 + lane;
    int nb = (s < upto) ? seq_blocks(a.pt.kv_lens[s], a.sm.window) : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) nb += __shfl_xor(nb, off);
    total += nb;
  }
  return uniform(total);
}

__device__ __forceinline__ int blocks_per_wave(const DecodeArgs& a, int total_blocks) {
  // never fewer than the even share: the grid has exactly num_wgs workgroups
  const int even = (total_blocks + a.num_wgs - 1) / a.num_wgs;
  const int floor_ = a.forced_blocks_per_wave > 0 ? a.forced_blocks_per_wave : a.min_blocks_per_wave;
  return max(floor_, even);
}

// sequence that holds linear block x (x < total): first s with (blocks of [0, s]) * units > x
__device__ __forceinline__ void locate_block(const DecodeArgs& a, int x, int units, int lane, int& seq,
                                             int& seq_first_block) {
  int base = 0;
  seq = a.num_rows - 1;
  seq_first_block = 0;
  for (int s0 = 0; s0 < a.num_rows; s0 += 64) {
    const int s = s0 + lane;
    const int nb = (s < a.num_rows) ? seq_blocks(a.pt.kv_lens[s], a.sm.window) : 0;
    const int incl = wave_inclusive_scan(nb, lane);
    const uint64_t hit = __builtin_amdgcn_ballot_w64((base + incl) * units > x);
    if (hit != 0) {
      const int first = __builtin_ctzll(hit);
      seq = s0 + first;
      seq_first_block = uniform((base + __shfl(incl - nb, first)) * units);
      return;
    }
    base += uniform(__shfl(incl, 63));
  }
}

// Wave-uniform facts of one decode row.
struct RowMeta {
  int seq;
  int kv_len;
  int nb;         // its 32-token blocks (0: nothing to read)
  int64_t page0;  // index of its first page id in page_indices
  int tq;         // its query token
};

struct RowLoads {  // the three words of a row, as loaded
  int kv_len, cu_kv, tq;
};

__device__ __forceinline__ RowLoads row_issue_scalar(const DecodeArgs& a, int seq) {
  RowLoads r;
  r.kv_len = scalar_load_i32(a.pt.kv_lens + seq);
  r.cu_kv = a.pt.cu_kv_lens ? scalar_load_i32(a.pt.cu_kv_lens + seq) : 0;
  r.tq = scalar_load_i32(a.pt.cu_q_lens + seq);
  return r;
}

__device__ __forceinline__ RowMeta row_resolve(const DecodeArgs& a, int seq, const RowLoads& r) {
  RowMeta m;
  m.seq = seq;
  m.kv_len = r.kv_len;
  m.nb = seq_blocks(r.kv_len, a.sm.window);
  m.page0 = a.pt.cu_kv_lens ? (int64_t)(r.cu_kv / a.pt.page_size) : (int64_t)seq * a.pt.pages_per_seq;
  m.tq = r.tq;
  return m;
}

// The balanced plan's window of a row's page ids (copy_page_window), looked up with a uniform LDS read
// when pages hold whole blocks and with one LDS read per lane and token row when they are smaller:
// the steady state of a wave issues no small dependent global loads at all, and because no
// register ever waits for the copy, the compiler never drains the vector-memory queue for it.
struct PageWindow {
  int32_t* lds;  // ids of this wave: 64 (whole blocks per page, one uniform lookup per block) or kWinSmallPages
  int first;     // slot of entry 0
};

template <int ENTRIES>
__device__ __forceinline__ void request_window(const DecodeArgs& a, const RowMeta& row, PageWindow& w,
                                               int first_slot, int page_shift, int lane) {
  w.first = first_slot;
  const int last_tok = max(row.kv_len - 1, 0);
  const int last_slot = page_shift >= 0 ? (last_tok >> page_shift) : (last_tok / a.pt.page_size);
  copy_page_window<ENTRIES>(a.pt.page_indices + row.page0, last_slot, w.lds, first_slot, lane);
}

// One piece of work of a wave: tokens of one (row, kv head, group of 16 query heads).
struct Piece {
  RowMeta row;
  int hk, rg;
  int t_lo;     // first visible token (sliding window)
  int t_first;  // first token of the piece (a multiple of 32 past the window's first block)
  int nblk;     // its 32-token blocks
  bool final_rows;
  float ks, vs;  // scales of the kv head's keys and values (asked for with the piece, a block before it begins)
};

// The wave that arrives last at a cut unit merges it.  A unit (row, kv head, group of 16 query
// heads) whose blocks n workgroups share leaves n groups of 16 partial rows; each wave, once its
// rows are written and fenced, adds one to the unit's arrival word, and the wave that brings it
// to n reads all n groups back and writes the 16 finished rows.  The word carries the call's
// generation in its upper 48 bits: a word left by another call (or by nothing: the memory is
// never cleared) counts as zero, and the merging wave sets the count back to zero so that a
// replay of the same launch with the same generation starts clean.
//
// A wave has at most two cut units, the first and the last piece of its share, and merges what
// falls to it after its last block: the registers of the block pipeline are free by then, so
// four groups of partial rows are in flight at a time, and no other wave waits for the rows.
struct PendingMerge {
  int n;  // 0: nothing to merge
  int w_first;
  int64_t first_block;
  int tq, head0, rows;
  unsigned long long* ctr;
};

// Every access is a device-scope atomic (relaxed): it reads what the other waves wrote through,
// whatever this part of the GPU still caches of an earlier call.  Lanes: dims 2 lane, 2 lane + 1
// of each of the 16 rows; lane r < 16 also owns the (max, sum) of row r.
__device__ __forceinline__ float load_agent(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void load2_agent(const float* p, float& x, float& y) {
  const unsigned long long v = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
  x = __uint_as_float((uint32_t)v);
  y = __uint_as_float((uint32_t)(v >> 32));
}

__device__ __forceinline__ void merge_unit(const DecodeArgs& a, const PendingMerge& pm, int pw, int wave, int nw,
                                           unsigned long long generation, int lane) {
  const int n = pm.n;
  const int r = lane & 15;
  auto slot16 = [&](int j) -> int64_t {
    const int wj = pm.w_first + min(j, n - 1);
    const int part = ((int64_t)wj * pw >= pm.first_block) ? 0 : 1;
    return (((int64_t)wj * nw + wave) * 2 + part) * 16;
  };
  float mstar = -INFINITY;
  for (int j = 0; j < n; ++j) mstar = fmaxf(mstar, load_agent(a.ws_ml + (slot16(j) + r) * 2));
  float den = 0.f;
  float acc[16][2];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i][0] = acc[i][1] = 0.f;
  for (int j0 = 0; j0 < n; j0 += 4) {  // four groups of partial rows in flight
    float o[4][16][2];
    float wgt[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t s = slot16(j0 + u);
#pragma unroll
      for (int i = 0; i < 16; ++i) load2_agent(a.ws_o + (s + i) * 128 + 2 * lane, o[u][i][0], o[u][i][1]);
      float mj, lj;
      load2_agent(a.ws_ml + (s + r) * 2, mj, lj);
      wgt[u] = (j0 + u < n) ? fast_exp2(mj - mstar) : 0.f;  // a repeated group counts nothing
      den += lj * wgt[u];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float wu = __shfl(wgt[u], i);
        acc[i][0] += o[u][i][0] * wu;
        acc[i][1] += o[u][i][1] * wu;
      }
  }
  const float inv_r =
      a.sm.sink ? sink_inverse(mstar, den, sink_logit(a.sm.sink, a.sm.round_logits, pm.head0 + min(r, pm.rows - 1)))
                : 1.0f / den;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float inv = __shfl(inv_r, i);
    if (i < pm.rows) {
      uint32_t* op = reinterpret_cast<uint32_t*>(a.out + ((int64_t)pm.tq * a.Hq + pm.head0 + i) * a.q_dim + 2 * lane);
      if (2 * lane < a.q_dim) *op = pack_bf16x2(acc[i][0] * inv, acc[i][1] * inv);
    }
  }
  if (lane == 0) __hip_atomic_store(pm.ctr, generation << 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// grid = num_wgs workgroups of NW = waves_per_wg waves.
//
// A wave treats its share as one stream of blocks: the block prefetched behind the last block of
// a piece is the first block of the next piece, the next row's lengths are fetched as scalar
// loads while the current piece streams, its page ids arrive as one window load and its queries
// are requested right behind that first block.  A piece border costs no round trip to memory,
// and neither does a block: under load a small dependent load waits behind megabytes of queued
// KV traffic (10 us and more), so there are none after the first block.
// e4m3: a block is half the bytes of a bf16 one and takes as long to work on, so one block ahead leaves the queue short (a block
// per 1.36 us and wave where the compute alone takes 1.0).  Its operands are converted into registers of their own first thing, and
// the block after next goes into the registers that this empties, across the borders of pieces: 64 rows of 1000..8000 tokens x 8
// heads on 16-token pages 124 -> 114 us, 128 rows of 1024..8192 x 8 heads on 64-token pages 204.7 -> 202.3 (the same without its compute: 2 % less).
// bf16 is bound by memory either way, and so has one block ahead.
// New tokens (a.new_k) are taken where pages hold whole blocks or halves.  (bf16: registers of one wave per SIMD, which is what is resident.)
template <int MT, bool FP8, Pages PG, bool CAP, bool MERGE, bool HALF>
__device__ __forceinline__ void decode_balanced(const DecodeArgs& a_in) {
  DecodeArgs a = a_in;  // static-shape mode: the number of decode rows comes from the device
  if (a.dist) a.num_rows = min(a.num_rows, scalar_load_i32(a.dist));
  if (a.num_rows <= 0) return;
  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int nw = a.waves_per_wg;
  const int wg = blockIdx.x;
  const int w = wg * nw + wave;
  const int row_groups = (a.G + 15) / 16;
  const int head_groups = (a.Hkv + nw - 1) / nw;
  const int units = head_groups * row_groups;
  const int page_size = a.pt.page_size;
  const int page_shift = ((page_size & (page_size - 1)) == 0) ? (31 - __builtin_clz(page_size)) : -1;

  // ---- one pass over the rows: lengths, page offsets and query tokens of rows 0..63 stay in
  // registers (most batches end there), the rest only adds to the total
  int kv0 = 0, cu0 = 0, tq0 = 0;
  if (lane < a.num_rows) {
    kv0 = a.pt.kv_lens[lane];
    cu0 = a.pt.cu_kv_lens ? a.pt.cu_kv_lens[lane] : 0;
    tq0 = a.pt.cu_q_lens[lane];
  }
  const int nb0 = seq_blocks(kv0, a.sm.window);
  const int incl0 = wave_inclusive_scan(nb0, lane);
  int total_rows = uniform(__shfl(incl0, 63));
  for (int s0 = 64; s0 < a.num_rows; s0 += 64) {
    const int s = s0 + lane;
    int nb = (s < a.num_rows) ? seq_blocks(a.pt.kv_lens[s], a.sm.window) : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) nb += __shfl_xor(nb, off);
    total_rows += uniform(nb);
  }
  const int total = total_rows * units;
  const int pw = blocks_per_wave(a, total);
  if (wg == 0 && wave == 0) {
    // the merge pass looks its rows up in this prefix sum instead of scanning again
    if (lane < a.num_rows) a.cu_blocks[lane + 1] = incl0;
    int base = uniform(__shfl(incl0, 63));
    for (int s0 = 64; s0 < a.num_rows; s0 += 64) {
      const int s = s0 + lane;
      const int nb = (s < a.num_rows) ? seq_blocks(a.pt.kv_lens[s], a.sm.window) : 0;
      const int incl = wave_inclusive_scan(nb, lane);
      if (s < a.num_rows) a.cu_blocks[s + 1] = base + incl;
      base += uniform(__shfl(incl, 63));
    }
    if (lane == 0) a.cu_blocks[0] = 0;
  }
  if ((int64_t)wg * pw >= total) return;
  int x = wg * pw;
  const int x_end = min(total, x + pw);
  const int x_first = x;

  // ---- the row that holds block x
  RowMeta row;
  int row_first;  // linear index of the row's first block
  {
    const uint64_t hit = __builtin_amdgcn_ballot_w64(incl0 * units > x);
    if (hit != 0) {
      const int first = __builtin_ctzll(hit);
      RowLoads rl;
      rl.kv_len = __builtin_amdgcn_readlane(kv0, first);
      rl.cu_kv = __builtin_amdgcn_readlane(cu0, first);
      rl.tq = __builtin_amdgcn_readlane(tq0, first);
      row = row_resolve(a, first, rl);
      row_first = uniform(__builtin_amdgcn_readlane(incl0 - nb0, first) * units);
    } else {
      int seq;
      locate_block(a, x, units, lane, seq, row_first);
      seq = uniform(seq);
      row = row_resolve(a, seq, row_issue_scalar(a, seq));
    }
  }

  auto make_piece = [&](const RowMeta& r, int unit, int blk, int take) {
    Piece p;
    p.row = r;
    const int hg = unit / row_groups;
    p.rg = unit - hg * row_groups;
    // a head group may reach past the last kv head: such a wave repeats the last head and its
    // result is dropped
    p.hk = hg * nw + wave;
    p.t_lo = (a.sm.window > 0) ? max(0, r.kv_len - a.sm.window) : 0;
    p.t_first = (p.t_lo & ~(kBlk - 1)) + blk * kBlk;
    p.nblk = take;
    p.final_rows = (blk == 0) && (take == r.nb);
    const int hk = min(p.hk, a.Hkv - 1);
    p.ks = a.k_scale ? scalar_load_f32(a.k_scale + hk) : 1.0f;
    p.vs = a.v_scale ? scalar_load_f32(a.v_scale + hk) : 1.0f;
    return p;
  };
  auto view_of = [&](const RowMeta& r, int hk) {
    SeqView sv;
    sv.page_size = page_size;
    sv.page_shift = page_shift;
    sv.last_tok = r.kv_len - 1;
    sv.pages = a.pt.page_indices + r.page0;
    sv.fresh_first = (PG != kLanes && a.new_k) ? r.kv_len - 1 : kNoFresh;
    sv.fresh_row = r.tq * a.Hkv + hk;
    return sv;
  };
  auto slot_of_tok = [&](int tok) { return page_shift >= 0 ? (tok >> page_shift) : (tok / page_size); };
  // ids of the pages that hold block tb of a row
  auto pages_in = [&](const PageWindow& pwn, const SeqView& v, int tb) -> BlockPages {
    BlockPages p = {};
    if constexpr (PG != kLanes) p.lo = uniform(pwn.lds[uniform(slot_of_tok(tb) - pwn.first)]);
    if constexpr (PG == kHalves) p.hi = uniform(pwn.lds[uniform(slot_of_tok(min(tb + 16, v.last_tok)) - pwn.first)]);
    return p;
  };
  Piece cur;
  {
    const int r = x - row_first;
    const int unit = r / row.nb;
    const int blk = r - unit * row.nb;
    cur = make_piece(row, unit, blk, min(row.nb - blk, x_end - x));
  }
  int cur_unit = (x - row_first) / row.nb;
  constexpr int kWin = PG == kBlocks ? 64 : kWinSmallPages;
  __shared__ int32_t lds_windows[4][2][kWin];  // [wave][current / next piece][entry]
  PageWindow win = {lds_windows[wave][0], 0};
  PageWindow nwin = {lds_windows[wave][1], 0};
  auto request = [&](KvRegs<FP8>& r, const SeqView& v, int of_head, const PageWindow& pwn, int tb, bool wanted) __attribute__((always_inline)) {
    load_cached_block<FP8, PG, HALF>(r, a, v, a.kv.k_base + (int64_t)of_head * a.kv.head_stride, a.kv.v_base + (int64_t)of_head * a.kv.head_stride,
                                     tb, pages_in(pwn, v, tb), wanted, c, g, pwn.lds, pwn.first);
  };
  request_window<kWin>(a, cur.row, win, slot_of_tok(cur.t_first), page_shift, lane);
  constexpr bool kTwo = FP8 && PG != kLanes;  // two blocks ahead
  u32x4_t qB[MT][4], q_next[MT][4];
  load_queries<MT, FP8>(a, cur.row.tq, min(cur.hk, a.Hkv - 1), cur.rg * 16 * MT, c, g, qB);
  wait_all_loads();  // the window (and the queries behind it)

  // ---- the piece at hand, and what is known of the one behind it: the next unit of the same row, or the first unit of the
  // next row that has any block (has_next guarantees there is one)
  KvRegs<FP8> ra, rb;
  int hk, i;  // its kv head, its next block
  SeqView sv;
  ScoreOpts so;
  NewTokenRegs<FP8, HALF> fresh;
  f32x4_t acc[MT][8];
  float m[MT], l[MT];
  bool has_next, next_row;
  int nseq;
  RowLoads nl;
  Piece nxt;
  auto begin_piece = [&]() __attribute__((always_inline)) {
    hk = min(cur.hk, a.Hkv - 1);
    sv = view_of(cur.row, hk);
    requantise_queries<MT, FP8>(a, qB);
    const float temp = xai_factor(cur.row.kv_len - 1, a.sm.xai_len);  // the one query sits at kv_len - 1
    const float scale = a.sm.sm_scale * cur.ks * (a.sm.q_scale > 0.f ? a.sm.q_scale : 1.0f);
    so.scale2 = scale * kLog2e * temp;
    so.general.set(a.sm, scale, temp);
    so.mask2 = fmaxf(a.sm.mask_value * kLog2e, -3.0e38f);
    so.t_lo = cur.t_lo;
    so.kv_len = cur.row.kv_len;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      m[mt] = -INFINITY;
      l[mt] = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[mt][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    has_next = x + cur.nblk < x_end;
    next_row = has_next && (cur_unit == units - 1);
    nseq = cur.row.seq + 1;
    nl = RowLoads{0, 0, 0};
    if (next_row) nl = row_issue_scalar(a, nseq);
    nxt = cur;
    fresh.on = PG != kLanes && a.new_k && cur.t_first + cur.nblk * kBlk > sv.last_tok;
    if (fresh.on) fresh.load(a, sv, c, g);
    i = 0;
  };
  PendingMerge pm_first = {}, pm_last = {};
  bool done = false;
  bool late = false;  // (two ahead) the piece's first block has not been asked for: the piece before was one block

  // One block: the one behind it is requested, then it is worked on; a piece's rows are written behind its last one.
  // false: nothing is left.
  auto step = [&](KvRegs<FP8>& use, KvRegs<FP8>& fill) __attribute__((always_inline)) -> bool {
    const int tb = cur.t_first + i * kBlk;
    const bool last = (i + 1 == cur.nblk);
    // resolved one block into the piece when it has more than one block, at once otherwise
    const int resolve_at = cur.nblk > (kTwo ? 2 : 1) ? 1 : 0;
    if (has_next && i == resolve_at) {
      RowMeta nrow = cur.row;
      int nunit = cur_unit + 1;
      if (next_row) {
        nrow = row_resolve(a, nseq, nl);
        while (nrow.nb == 0) {  // rows without tokens (padding)
          ++nseq;
          nrow = row_resolve(a, nseq, row_issue_scalar(a, nseq));
        }
        nunit = 0;
      }
      const int x_next = x + cur.nblk;
      nxt = make_piece(nrow, nunit, 0, min(nrow.nb, x_end - x_next));
      request_window<kWin>(a, nrow, nwin, slot_of_tok(nxt.t_first), page_shift, lane);
      if constexpr (kTwo) load_queries<MT, FP8>(a, nxt.row.tq, min(nxt.hk, a.Hkv - 1), nxt.rg * 16 * MT, c, g, q_next);
    }
    if constexpr (kTwo) {
      if (rare(late)) {
        wait_all_loads();
        request(use, sv, hk, win, tb, true);
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0), by a name that the compiler counts by
        late = false;
      }
      if (rare(fresh.on && last)) fresh.put(use, sv.last_tok - tb, c, g);
      compute_block<MT, FP8, CAP, HALF, PG == kBlocks>(use, qB, acc, m, l, so, tb, g, [&]() __attribute__((always_inline)) {
        const int beyond = i + 2 - cur.nblk;  // block of the next piece, when not negative
        const bool here = beyond < 0, there = has_next && beyond >= 0 && beyond < nxt.nblk;
        const int t_ask = min(tb + 2 * kBlk, cur.t_first + (cur.nblk - 1) * kBlk);
        if (here && slot_of_tok(t_ask + (PG == kBlocks ? 0 : kBlk - 1)) - win.first >= kWin) {
          request_window<kWin>(a, cur.row, win, slot_of_tok(t_ask), page_shift, lane);
          wait_all_loads();
        }
        if (there && i <= resolve_at + 1) wait_all_loads();
        const int fhk = there ? min(nxt.hk, a.Hkv - 1) : hk;
        request(use, view_of(there ? nxt.row : cur.row, fhk), fhk, there ? nwin : win, there ? nxt.t_first + beyond * kBlk : t_ask, here || there);
      });
    } else {
      // the window moves on when the next block's last page lies beyond it
      if (!last && slot_of_tok(tb + kBlk + (PG == kBlocks ? 0 : kBlk - 1)) - win.first >= kWin) {
        request_window<kWin>(a, cur.row, win, slot_of_tok(tb + kBlk), page_shift, lane);
        wait_all_loads();
      }
      // The next piece's window was requested at block resolve_at, in front of that block's
      // prefetch.  Two blocks later a wait for younger loads has passed; earlier it has not.
      if (last && has_next && i <= resolve_at + 1) wait_all_loads();
      // The block to request now: the next one of this piece, the first one of the next piece, or (nothing left) one that is not
      // wanted.  What differs is chosen in scalars and the loads stand once, in no branch: with a way around them in the code the
      // compiler waits for all loads where it should wait for the block in use alone.
      {
        const bool ahead = last && has_next;
        const int fhk = ahead ? min(nxt.hk, a.Hkv - 1) : hk;
        request(fill, view_of(ahead ? nxt.row : cur.row, fhk), fhk, ahead ? nwin : win, ahead ? nxt.t_first : last ? tb : tb + kBlk, ahead || !last);
      }
      if (PG != kLanes && rare(fresh.on && last)) fresh.put(use, sv.last_tok - tb, c, g);
      compute_block<MT, FP8, CAP, HALF, PG == kBlocks>(use, qB, acc, m, l, so, tb, g);
    }
    ++i;
    if (!last) return true;

    if (PG != kLanes && fresh.on) {
      const int slot = slot_of_tok(sv.last_tok);
      fresh.store(a.kv, a.kv.k_base + (int64_t)hk * a.kv.head_stride, a.kv.v_base + (int64_t)hk * a.kv.head_stride,
                  uniform(win.lds[uniform(slot - win.first)]), sv.last_tok - slot * page_size, c, g);
    }
    if (cur.hk < a.Hkv) {
      PartDest dest;
      dest.final_rows = cur.final_rows;
      dest.by_head = false;
      dest.base = ((int64_t)w * 2 + (x == x_first ? 0 : 1)) * 16;
      write_rows<MT, MERGE>(a, acc, m, l, cur.row.tq, hk, cur.rg * 16 * MT, dest, cur.vs, c, g);
      if (MERGE && !cur.final_rows) {
        // the unit's first block in the linear order, and the workgroups that share the unit
        const int64_t first_block = (int64_t)x - (cur.t_first - (cur.t_lo & ~(kBlk - 1))) / kBlk;
        const int w_first = (int)(first_block / pw), w_last = (int)((first_block + cur.row.nb - 1) / pw);
        const unsigned long long n = (unsigned long long)(w_last - w_first + 1);
        unsigned long long* ctr = a.merge_counters + ((int64_t)cur.row.seq * units + cur_unit) * nw + wave;
        // this wave's rows, written through, have reached device scope before it arrives
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        int is_last = 0;
        if (lane == 0) {
          unsigned long long old = __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          for (;;) {
            const unsigned long long cnt = ((old >> 16) == a.generation) ? (old & 0xffffull) : 0ull;
            const unsigned long long neu = (a.generation << 16) | (cnt + 1);
            if (__hip_atomic_compare_exchange_strong(ctr, &old, neu, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT)) {
              is_last = (cnt + 1 == n) ? 1 : 0;
              break;
            }
          }
        }
        is_last = __builtin_amdgcn_readfirstlane(is_last);
        if (is_last) {
          PendingMerge& pm = (x == x_first) ? pm_first : pm_last;
          pm.n = (int)n;
          pm.w_first = w_first;
          pm.first_block = first_block;
          pm.tq = cur.row.tq;
          pm.head0 = hk * a.G + cur.rg * 16;
          pm.rows = min(16, a.G - cur.rg * 16);
          pm.ctr = ctr;
        }
      }
    }
    if (!has_next) {
      done = true;
      return false;
    }
    x += cur.nblk;
    cur_unit = next_row ? 0 : cur_unit + 1;
    late = cur.nblk == 1;
    cur = nxt;
    {  // the two LDS windows trade places
      const PageWindow t = win;
      win = nwin;
      nwin = t;
    }
    // the queries queue up right behind the piece's first block, which is already on its way
    if constexpr (kTwo) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int st = 0; st < 4; ++st) qB[mt][st] = q_next[mt][st];
    } else {
      load_queries<MT, FP8>(a, cur.row.tq, min(cur.hk, a.Hkv - 1), cur.rg * 16 * MT, c, g, qB);
    }
    begin_piece();
    return true;
  };
  begin_piece();
  request(ra, sv, hk, win, cur.t_first, true);
  if constexpr (kTwo) __builtin_amdgcn_sched_barrier(0);  // (the waits in the loop count on this order)
  if constexpr (kTwo) request(rb, sv, hk, win, min(cur.t_first + kBlk, cur.t_first + (cur.nblk - 1) * kBlk), cur.nblk > 1);
  if constexpr (kTwo) {
    // no way out between the two: the compiler would see one from there back to the top, with the first step's loads as the
    // youngest in flight, and wait for all of them.  A step behind the last block works on one that is not wanted.
    do {
      step(ra, rb);
      step(rb, ra);
    } while (!done);
  } else {
    while (step(ra, rb) && step(rb, ra)) {
    }
  }
  if (MERGE && (pm_first.n | pm_last.n)) {
    if (pm_first.n) merge_unit(a, pm_first, pw, wave, nw, a.generation, lane);
    if (pm_last.n) merge_unit(a, pm_last, pw, wave, nw, a.generation, lane);
  }
}

template <int MT, bool FP8, bool UNIFORM_PAGE, bool CAP, bool MERGE, bool HALF = false>
__global__ __launch_bounds__(256, FP8 ? 2 : 1) void rpa_decode_balanced_kernel(const DecodeArgs a) {
  decode_balanced<MT, FP8, UNIFORM_PAGE ? kBlocks : kLanes, CAP, MERGE, HALF>(a);
}

template <int MT, bool FP8, bool CAP, bool MERGE, bool HALF = false>
__global__ __launch_bounds__(256, FP8 ? 2 : 1) void rpa_decode_balanced_halves_kernel(const DecodeArgs a) {
  decode_balanced<MT, FP8, kHalves, CAP, MERGE, HALF>(a);
}

// Merge the n partial rows of one (decode row, query head) and write the finished row.
// slot_of(j) is the workspace slot of partial j.  One wave, 2 dims per lane.  Up to 16 partials
// (nearly always) everything is requested at once -- the (max, sum) pairs by lanes 0..n-1, the
// partial rows by all lanes, the row's query token before either -- so the merge costs one round
// trip to memory instead of three dependent ones.
// The merge kernels come in sizes, chosen by merge_size().  With the code for many partials and its LDS in the one that every
// small step runs, and a choice between 8 and 16 partials in front of the requests, a call of 5 rows of 64..512 tokens x 16 / 8
// heads took 9.82 us (replayed from a graph) and one of 8 rows x 8 / 2 heads 8.23; without them 9.77 and 8.15.
enum MergeSize {
  kMergeEight,    // one wave, at most 8 partials
  kMergeSixteen,  // one wave, at most 16
  kMergeAny,      // one wave, any number
  kMergeWide,     // four waves, any number
};
constexpr int kMergeWaves = 4;
constexpr int merge_threads(MergeSize size) { return size == kMergeWide ? 64 * kMergeWaves : 64; }

template <int N, int HD, typename SlotOf>
__device__ __forceinline__ void merge_few(const DecodeArgs& a, int n, int lane, SlotOf slot_of, float& mstar,
                                          float& den, float (&acc)[HD / 64]) {
  constexpr int kDpl = HD / 64;  // dims per lane
  typedef float fvec_t __attribute__((ext_vector_type(kDpl)));
  const int d = lane * kDpl;
  // (every lane loads: behind a branch on lane < n the compiler waits for the pair before it asks for the rows)
  const f32x2_t ml = *reinterpret_cast<const f32x2_t*>(a.ws_ml + slot_of(min(lane, n - 1)) * 2);
  fvec_t o[N];
#pragma unroll
  for (int u = 0; u < N; ++u) o[u] = *reinterpret_cast<const fvec_t*>(a.ws_o + slot_of(min(u, n - 1)) * HD + d);
  const float mj = lane < n ? ml[0] : -INFINITY, lj = ml[1];
  mstar = mj;
#pragma unroll
  for (int off = N / 2; off > 0; off >>= 1) mstar = fmaxf(mstar, __shfl_xor(mstar, off));
  mstar = __shfl(mstar, 0);
  const float wj = (lane < n) ? fast_exp2(mj - mstar) : 0.f;
  den = lj * wj;
#pragma unroll
  for (int off = N / 2; off > 0; off >>= 1) den += __shfl_xor(den, off);
  den = __shfl(den, 0);
#pragma unroll
  for (int e = 0; e < kDpl; ++e) acc[e] = 0.f;
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const float wu = __shfl(wj, u);  // 0 beyond n: the repeated last row does not count
#pragma unroll
    for (int e = 0; e < kDpl; ++e) acc[e] += o[u][e] * wu;
  }
}

// More than 16 partials (a few rows cut over the whole chip): the waves of the workgroup take 16 partial rows each in turn, and
// wave 0 adds what they have.  One wave with 32 rows at a time behind two passes over the references was a chain of up to
// seven round trips: 7 rows of 221 .. 6024 tokens x 8 heads 11.1 -> 6.0 us, 2 rows of
// 20000 .. 30000 x 8 heads 9.0 -> 4.8.  Returns whether this wave goes on to write.
template <int HD, int WAVES, typename SlotOf>
__device__ __forceinline__ bool merge_many(const DecodeArgs& a, int n, int lane, SlotOf slot_of, float& mstar, float& den,
                                           float (&acc)[HD / 64]) {
  constexpr int kDpl = HD / 64;
  typedef float fvec_t __attribute__((ext_vector_type(kDpl)));
  const int wave = WAVES > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  for (int b0 = 0; b0 < n; b0 += 256) {  // references and sums of 256 partials in one round trip
    float mj[4], lj[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = b0 + 64 * u + lane;
      mj[u] = -INFINITY;
      lj[u] = 0.f;
      if (j < n) {
        const int64_t slot = slot_of(j);
        mj[u] = a.ws_ml[slot * 2];
        lj[u] = a.ws_ml[slot * 2 + 1];
      }
    }
    float top = fmaxf(fmaxf(mj[0], mj[1]), fmaxf(mj[2], mj[3]));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) top = fmaxf(top, __shfl_xor(top, off));
    top = fmaxf(mstar, top);
    const float keep = b0 > 0 ? fast_exp2(mstar - top) : 0.f;
    mstar = top;
    den *= keep;
#pragma unroll
    for (int e = 0; e < kDpl; ++e) acc[e] *= keep;
    float wj[4], lsum = 0.f;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      wj[u] = b0 + 64 * u + lane < n ? fast_exp2(mj[u] - mstar) : 0.f;
      lsum += lj[u] * wj[u];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off);
    den += lsum;
    for (int j0 = b0 + wave * 16; j0 < min(n, b0 + 256); j0 += WAVES * 16) {
      const int part = (j0 - b0) >> 6, first = (j0 - b0) & 63;
      const float wp = part == 0 ? wj[0] : part == 1 ? wj[1] : part == 2 ? wj[2] : wj[3];
      fvec_t o[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) o[u] = *reinterpret_cast<const fvec_t*>(a.ws_o + slot_of(min(j0 + u, n - 1)) * HD + lane * kDpl);
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const float wu = __shfl(wp, first + u);  // 0 beyond n: the repeated last row does not count
#pragma unroll
        for (int e = 0; e < kDpl; ++e) acc[e] += o[u][e] * wu;
      }
    }
  }
  if constexpr (WAVES > 1) {
    __shared__ float sums[WAVES - 1][HD];
    if (wave > 0) {
#pragma unroll
      for (int e = 0; e < kDpl; ++e) sums[wave - 1][lane * kDpl + e] = acc[e];
    }
    __syncthreads();
    if (wave > 0) return false;
    for (int w = 0; w < WAVES - 1; ++w)
#pragma unroll
      for (int e = 0; e < kDpl; ++e) acc[e] += sums[w][lane * kDpl + e];
  }
  return true;
}

template <int HD, MergeSize SIZE, typename SlotOf>
__device__ __forceinline__ void merge_rows(const DecodeArgs& a, int tq, int head, int n, int lane, SlotOf slot_of) {
  constexpr int kDpl = HD / 64;  // dims per lane
  const int d = lane * kDpl;
  float mstar = -INFINITY, den = 0.f;
  float acc[kDpl];
#pragma unroll
  for (int e = 0; e < kDpl; ++e) acc[e] = 0.f;
  if constexpr (SIZE == kMergeEight) {
    merge_few<8, HD>(a, n, lane, slot_of, mstar, den, acc);
  } else if constexpr (SIZE == kMergeSixteen) {
    merge_few<16, HD>(a, n, lane, slot_of, mstar, den, acc);
  } else if (n <= 16) {
    if (SIZE == kMergeWide && threadIdx.x >= 64) return;
    if (n <= 8) merge_few<8, HD>(a, n, lane, slot_of, mstar, den, acc);
    else merge_few<16, HD>(a, n, lane, slot_of, mstar, den, acc);
  } else if (!merge_many<HD, merge_threads(SIZE) / 64>(a, n, lane, slot_of, mstar, den, acc)) {
    return;
  }
  const float inv = a.sm.sink ? sink_inverse(mstar, den, sink_logit(a.sm.sink, a.sm.round_logits, head)) : 1.0f / den;
  if (d >= a.q_dim) return;
  uint32_t* op = reinterpret_cast<uint32_t*>(a.out + ((int64_t)tq * a.Hq + head) * a.q_dim + d);
#pragma unroll
  for (int e = 0; e < kDpl; e += 2) op[e / 2] = pack_bf16x2(acc[e] * inv, acc[e + 1] * inv);
}

// The merge kernel for `rows` rows whose units are cut into `pieces` on average and `most` at most: more than a wave where there
// are many partials and few rows (idle waves of large launches cost more than they save).
MergeSize merge_size(const DecodeArgs& a, int64_t rows, int64_t pieces, int64_t most) {
  return most <= 8 ? kMergeEight : most <= 16 ? kMergeSixteen : pieces > 8 && rows * a.Hq <= 2048 ? kMergeWide : kMergeAny;
}

// Merge the partial rows of the balanced plan.  grid = (Hq * decode rows); block = merge_threads(SIZE).
template <MergeSize SIZE>
__global__ __launch_bounds__(merge_threads(SIZE)) void rpa_combine_balanced_kernel(const DecodeArgs a_in) {
  DecodeArgs a = a_in;  // static-shape mode: the number of decode rows comes from the device
  if (a.dist) a.num_rows = min(a.num_rows, scalar_load_i32(a.dist));
  const int seq = (int)(blockIdx.x / (unsigned)a.Hq);  // grid.x = Hq * rows, heads fastest
  const int head = (int)blockIdx.x - seq * a.Hq;
  if (seq >= a.num_rows) return;
  const int lane = threadIdx.x & 63;
  const int nw = a.waves_per_wg;
  const int row_groups = (a.G + 15) / 16;
  const int units = ((a.Hkv + nw - 1) / nw) * row_groups;
  // (what the merge has to know in one round trip)
  const int kv_len = scalar_load_i32(a.pt.kv_lens + seq), before = scalar_load_i32(a.cu_blocks + seq);
  const int total = scalar_load_i32(a.cu_blocks + a.num_rows) * units, tq = scalar_load_i32(a.pt.cu_q_lens + seq);
  const int nb = seq_blocks(kv_len, a.sm.window);
  if (nb == 0) return;
  const int pw = blocks_per_wave(a, total);
  const int hk = head / a.G, row = head - hk * a.G;
  const int unit = (hk / nw) * row_groups + row / 16;
  const int wv = hk % nw;
  const int first_block = before * units + unit * nb;
  const int w_first = first_block / pw, w_last = (first_block + nb - 1) / pw;
  if (w_first == w_last) return;  // one wave covered the unit and wrote the finished rows
  const int n = w_last - w_first + 1;
  const int r16 = row & 15;
  auto slot_of = [&](int j) -> int64_t {
    const int wj = w_first + j;  // workgroup
    // a workgroup's first piece of work goes to slot 0 of its waves: that is this unit iff it starts inside it
    const int part = ((int64_t)wj * pw >= first_block) ? 0 : 1;
    return (((int64_t)wj * nw + wv) * 2 + part) * 16 + r16;
  };
  merge_rows<128, SIZE>(a, tq, head, n, lane, slot_of);
}

// ---- head_dim 256 ---------------------------------------------------------------------------
// One wave per (query token, kv head, group of 16 query heads): a query token of a chunk is a
// decode row over the first kv_len - q_len + j + 1 tokens, so one kernel serves decode rows and
// prefill chunks alike.  The two 128-dim halves of a head reuse the register layouts and the
// loads of the 128-dim kernel (a half is 128 contiguous elements of the head's row); scores sum
// over both halves, each half has its own accumulators.  A chunk's tokens each stream the prefix
// again (chunks take the prefill kernel unless a switch sends them here).
// grid = (token rows, Hkv, row groups of 16 query heads); block = one wave.
// With the composition on the device (a.dist) seq_end is only a bound: dist_role 1 = the decode partition
// [0, dist[0]), 2 = everything behind it [dist[0], dist[2]) (custom-mask calls: [0, dist[2])).
template <bool FP8, Pages PG>
__global__ __launch_bounds__(64, FP8 ? 2 : 1) void rpa_rows256_kernel(const DecodeArgs a, int seq_begin, int seq_end, int dist_role) {
  if (a.dist && dist_role == 1) {
    seq_end = min(seq_end, scalar_load_i32(a.dist));
  } else if (a.dist && dist_role == 2) {
    seq_begin = (a.sm.mask_mode == 1) ? 0 : min(seq_end, scalar_load_i32(a.dist));
    seq_end = min(seq_end, scalar_load_i32(a.dist + 2));
  }
  if (seq_end <= seq_begin) return;
  const int lane = threadIdx.x;
  const int c = lane & 15, g = lane >> 4;
  const int rg = blockIdx.z, hk = blockIdx.y;
  // decode rows may be cut into max_splits pieces of `chunk` tokens (one token per row then, and
  // row = sequence); partial rows go to the workspace in the fixed plan's layout
  const int nsplit = max(a.max_splits, 1);
  // Pieces outermost, rows and heads turned against the workgroup's number: workgroups go to the XCDs by number, and with
  // the pieces of a row next to one another an XCD got the same piece of every row, mostly an empty one where few rows
  // are long (180 rows of 500..3000 e4m3 tokens x 8 heads, two pieces: 392 -> 277 us).
  const int nrows = gridDim.x / nsplit, split = blockIdx.x / nrows;
  const int tok_row = (blockIdx.x + split + hk) % nrows + a.pt.cu_q_lens[seq_begin];
  if (tok_row >= a.pt.cu_q_lens[seq_end]) return;
  const int seq = owner_of_token(a.pt.cu_q_lens, seq_end, tok_row);
  const int q0 = a.pt.cu_q_lens[seq];
  const int q_len = a.pt.cu_q_lens[seq + 1] - q0;
  const int kv_len = a.pt.kv_lens[seq];
  const int qpos = kv_len - q_len + (tok_row - q0);
  // tokens this row sees: [t_lo, t_hi)
  const int t_hi = (a.sm.mask_mode == 0) ? qpos + 1 : kv_len;
  if (t_hi <= 0) return;
  const int t_lo = (a.sm.window > 0) ? max(0, qpos - a.sm.window + 1) : 0;
  // the caller's own mask: one i32 per (query token, kv token), rows kv_len wide or padded to whole pages
  const int32_t* mask_row = nullptr;
  if (a.sm.mask_mode == 1) {
    const int width = a.sm.mask_rows_page_aligned ? (a.pt.cu_kv_lens[seq + 1] - a.pt.cu_kv_lens[seq]) : kv_len;
    mask_row = a.sm.custom_mask + a.sm.cu_mask_lens[seq] + (int64_t)(tok_row - q0) * width;
  }

  SeqView sv;
  sv.page_size = a.pt.page_size;
  sv.page_shift = ((sv.page_size & (sv.page_size - 1)) == 0) ? (31 - __builtin_clz(sv.page_size)) : -1;
  sv.last_tok = t_hi - 1;
  sv.fresh_first = kNoFresh;
  sv.pages = a.pt.page_indices + (a.pt.cu_kv_lens ? (a.pt.cu_kv_lens[seq] / a.pt.page_size)
                                                  : (int64_t)seq * a.pt.pages_per_seq);
  constexpr int kHalfB = FP8 ? 128 : 256;  // bytes of 128 cached elements
  const char* kh = a.kv.k_base + (int64_t)hk * a.kv.head_stride;
  const char* vh = a.kv.v_base + (int64_t)hk * a.kv.head_stride;

  // ---- Q^T operands: column c = query head (16 rg + c) of this kv head, both halves ----
  const int row = rg * 16 + c;
  u32x4_t qB[2][4];
  {
    const uint16_t* qp = a.q + ((int64_t)tok_row * a.Hq + (int64_t)hk * a.G + min(row, a.G - 1)) * a.q_dim;
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const int d0 = hf * 128 + (FP8 ? g * 32 + st * 8 : st * 32 + g * 8);
        qB[hf][st] = ld_query(qp, d0, a.q_dim);
        if (a.sm.q_scale > 0.f) qB[hf][st] = requantise_q(qB[hf][st], a.sm.q_scale, FP8);
      }
  }
  const float scale = a.sm.sm_scale * (a.k_scale ? a.k_scale[hk] : 1.0f) * (a.sm.q_scale > 0.f ? a.sm.q_scale : 1.0f);
  LogitOpts general;
  const float temp = xai_factor(qpos, a.sm.xai_len), cap = a.sm.soft_cap, inv_cap = cap != 0.f ? 1.0f / cap : 0.f;
  general.set(a.sm, scale, temp);
  const float mask2 = fmaxf(a.sm.mask_value * kLog2e, -3.0e38f);

  f32x4_t acc[2][8];
#pragma unroll
  for (int hf = 0; hf < 2; ++hf)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[hf][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  int tb_begin = t_lo & ~(kBlk - 1), tb_end = t_hi;
  if (nsplit > 1) {
    tb_begin += split * a.chunk;
    if (tb_begin >= t_hi) return;  // the merge pass knows how many pieces a row has
    if (split < nsplit - 1) tb_end = min(t_hi, tb_begin + a.chunk);
  }
  // The row's new token, from the caller's rows into its slot, by every wave that reads it, in front of everything that the wave reads
  // (the same bytes from each; its loads follow its own stores).  A round trip to memory for the waves of a row's last piece; as a launch
  // in front it was 4 us for any batch: 5 rows of 1396..8992 e4m3 tokens x 2 heads 22.2 -> 17.6 us, 14 behind a window of 512 13.6 -> 10.8.
  if (a.new_k && tb_end == t_hi && tb_begin < tb_end) {
    constexpr int kRow = 2 * kHalfB;
    const int src_row = a.q_dim * (FP8 ? 1 : 2);  // the rest of a cached row is zero
    const int at = (lane & 31) * 16;
    const int slot = page_slot_of(sv, sv.last_tok);
    const int64_t to = (int64_t)scalar_load_i32(sv.pages + __builtin_amdgcn_readfirstlane(slot)) * a.kv.page_stride +
                       (int64_t)(sv.last_tok - slot * sv.page_size) * a.kv.tok_stride + at;
    const int64_t from = ((int64_t)tok_row * a.Hkv + hk) * src_row + at;
    u32x4_t x = {0u, 0u, 0u, 0u};
    if (at < src_row) x = ld16((lane < 32 ? a.new_k : a.new_v) + from);
    if (at < kRow) st16(const_cast<char*>(lane < 32 ? kh : vh) + to, x);
    wait_all_loads();  // (and stores)
  }
  // kLanes: the lanes look their token rows' pages up in an LDS window of the row's page
  // ids (see decode_segment) instead of fetching them from memory in front of every block
  __shared__ int32_t win_ids[PG != kLanes ? 1 : kWinSmallPages];
  const int32_t* win = nullptr;
  int win_first = 0;
  // The registers of a block's K rows are free behind the first product, those of its V rows behind the second: the next
  // block's rows are requested into them there, so that half a block is always on its way and no register is needed
  // twice (two whole blocks do not fit beside the 64 accumulators at two waves per SIMD, which
  // e4m3 keeps; bf16 needs one wave's registers).
  // 32 rows of 8000..16000 tokens x 8 heads: bf16 642 -> 567 us, e4m3 on 16-token pages 431 -> 302 (e4m3 on 64-token pages
  // was level at 300); 100 rows, window 512, e4m3 46.2 -> 31; 8 rows of 300..3000 36.9 -> 26.
  // Not bf16 on kLanes pages, where every half would begin with ids from LDS and an address per lane and load: the loop
  // there is the plain one, options asked per score (32 rows 575 us, 589 with half a block ahead; 64 rows of 1000 .. 8000 521
  // and 534).
  constexpr bool kAhead = FP8 || PG != kLanes;
  BlockPages page = {}, page_next = {};
  auto page_of = [&](int tb) __attribute__((always_inline)) {
    BlockPages p = {};
    p.lo = scalar_load_i32(sv.pages + page_slot_of(sv, min(tb, sv.last_tok)));
    if constexpr (PG == kHalves) p.hi = scalar_load_i32(sv.pages + page_slot_of(sv, min(tb + 16, sv.last_tok)));
    return p;
  };
  KvRegs<FP8> r0, r1;
  auto locate = [&](int tb) __attribute__((always_inline)) {
    if constexpr (PG != kLanes) {
      page = page_next;
      page_next = page_of(tb + kBlk);
    } else if (!win || page_slot_of(sv, min(tb + kBlk - 1, sv.last_tok)) - win_first >= kWinSmallPages) {
      win_first = __builtin_amdgcn_readfirstlane(page_slot_of(sv, tb));
      copy_page_window<kWinSmallPages>(sv.pages, page_slot_of(sv, sv.last_tok), win_ids, win_first, lane);
      wait_all_loads();
      win = win_ids;
    }
  };
  auto request_k = [&](int tb) __attribute__((always_inline)) {
    locate(tb);
    load_block<FP8, PG, PG == kLanes, false, false, kOnlyK>(r0, a, sv, kh, vh, tb, page, c, g, win, win_first);
    load_block<FP8, PG, PG == kLanes, false, false, kOnlyK>(r1, a, sv, kh + kHalfB, vh + kHalfB, tb, page, c, g, win, win_first);
  };
  auto request_v = [&](int tb) __attribute__((always_inline)) {
    load_block<FP8, PG, PG == kLanes, false, false, kOnlyV>(r0, a, sv, kh, vh, tb, page, c, g, win, win_first);
    load_block<FP8, PG, PG == kLanes, false, false, kOnlyV>(r1, a, sv, kh + kHalfB, vh + kHalfB, tb, page, c, g, win, win_first);
  };
  if constexpr (PG != kLanes) page_next = page_of(tb_begin);
  if (kAhead && tb_begin < tb_end) {
    request_k(tb_begin);
    request_v(tb_begin);
  }
  for (int tb = tb_begin; tb < tb_end; tb += kBlk) {
    const bool more = kAhead && tb + kBlk < tb_end;
    if constexpr (!kAhead) {
      locate(tb);
      load_block<FP8, PG, PG == kLanes>(r0, a, sv, kh, vh, tb, page, c, g, win, win_first);
      load_block<FP8, PG, PG == kLanes>(r1, a, sv, kh + kHalfB, vh + kHalfB, tb, page, c, g, win, win_first);
    }
    f32x4_t s[2];
    {
      u32x4_t kA[2][4];
      k_operands<FP8>(r0, kA);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        s[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < 4; ++st) s[b] = mfma16(kA[b][st], qB[0][st], s[b]);
      }
      k_operands<FP8>(r1, kA);
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int st = 0; st < 4; ++st) s[b] = mfma16(kA[b][st], qB[1][st], s[b]);
    }
    if (more) request_k(tb + kBlk);
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = s[i >> 2][i & 3];
    if constexpr (kAhead) {
      general.apply(x);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float v = x[i] * scale;
        if (cap != 0.f) v = soft_cap_f(v, cap, inv_cap);
        v = v * temp;
        if (general.round_mode) v = round_logit(v, general.round_mode);
        x[i] = v * kLog2e;
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int tok = tb + tok_slot(g, i);
      bool dead = tok >= tb_end || tok < t_lo;
      if (mask_row && !dead) dead = mask_row[tok] < 1;
      if (dead) x[i] = mask2;
    }
    const float mx = swap_max(swap16_max(max8(x)));
    const float m_new = fmaxf(m, mx);
    const float alpha = fast_exp2(m - m_new);
    float p[8], ps = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      p[i] = fast_exp2(x[i] - m_new);
      ps += p[i];
    }
    l = l * alpha + ps;
    m = m_new;
    const u32x4_t pB = u32x4_t{pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3]), pack_bf16x2(p[4], p[5]),
                               pack_bf16x2(p[6], p[7])};
    if (kAhead && (!FP8 || __builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0)) {  // as in compute_block: a maximum seldom moves
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[hf][j] = acc[hf][j] * alpha;
    }
    {
      u32x4_t vA[8];
      v_operands<FP8>(r0, vA);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[0][j] = mfma16(vA[j], pB, kAhead ? acc[0][j] : acc[0][j] * alpha);
      v_operands<FP8>(r1, vA);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[1][j] = mfma16(vA[j], pB, kAhead ? acc[1][j] : acc[1][j] * alpha);
    }
    if (more) request_v(tb + kBlk);
  }

  // ---- epilogue: lane (c, g) holds q row c, dims 128 hf + 32g + 8r + j in acc[hf][j][r] ----
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (row >= a.G) return;
  const int head = hk * a.G + row;
  const float vs = a.v_scale ? a.v_scale[hk] : 1.0f;
  if (nsplit > 1) {
    const int64_t slot = ((int64_t)seq * nsplit + split) * a.Hq + head;
    float* wo = a.ws_o + slot * 256 + g * 32;
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        f32x4_t w0 = {acc[hf][0][r] * vs, acc[hf][1][r] * vs, acc[hf][2][r] * vs, acc[hf][3][r] * vs};
        f32x4_t w1 = {acc[hf][4][r] * vs, acc[hf][5][r] * vs, acc[hf][6][r] * vs, acc[hf][7][r] * vs};
        *reinterpret_cast<f32x4_t*>(wo + hf * 128 + r * 8) = w0;
        *reinterpret_cast<f32x4_t*>(wo + hf * 128 + r * 8 + 4) = w1;
      }
    if (g == 0) {
      a.ws_ml[slot * 2 + 0] = m;
      a.ws_ml[slot * 2 + 1] = l;
    }
    return;
  }
  const float inv = a.sm.sink ? vs * sink_inverse(m, l, sink_logit(a.sm.sink, a.sm.round_logits, head)) : vs / l;
  uint16_t* op = a.out + ((int64_t)tok_row * a.Hq + head) * a.q_dim + g * 32;
#pragma unroll
  for (int hf = 0; hf < 2; ++hf)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (hf * 128 + g * 32 + r * 8 >= a.q_dim) break;
      u32x4_t w;
#pragma unroll
      for (int jp = 0; jp < 4; ++jp) w[jp] = pack_bf16x2(acc[hf][2 * jp][r] * inv, acc[hf][2 * jp + 1][r] * inv);
      st16(op + hf * 128 + r * 8, w);
    }
}

// Merge the split partials: out = sum_j o_j 2^(m_j - m*) / sum_j l_j 2^(m_j - m*).
// grid = (Hq * decode rows); block = merge_threads(SIZE), 2 dims per lane (D = 128).  Lane j
// first fetches (m_j, l_j) of split j, the wave reduces m* and the denominator
// with shuffles, then the weights are broadcast lane by lane while the partial
// rows stream in with independent loads.
template <int HD, MergeSize SIZE>
__global__ __launch_bounds__(merge_threads(SIZE)) void rpa_combine_kernel(const DecodeArgs a) {
  const int index = (int)(blockIdx.x / (unsigned)a.Hq);  // grid.x = Hq * rows, heads fastest
  const int head = (int)blockIdx.x - index * a.Hq;
  RowRef row;
  if (!fixed_row(a, index, row)) return;
  const int lane = threadIdx.x & 63;
  const int t0 = first_block_token(row.kv_len, a.sm.window);
  const int n = min(a.max_splits, (row.kv_len - t0 + a.chunk - 1) / a.chunk);
  if (n <= 0) return;
  const int64_t base = ((int64_t)index * a.max_splits) * a.Hq + head;
  merge_rows<HD, SIZE>(a, row.tq, head, n, lane, [&](int j) -> int64_t { return base + (int64_t)j * a.Hq; });
}

// One thread copies one 16-byte piece of one gathered row.
__global__ __launch_bounds__(256) void rpa_gather_kernel(const GatherArgs a) {
  const int kv_len = min(a.pt.kv_lens[a.seq], a.max_tokens);
  const int pieces = a.row_bytes / 16;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t total = (int64_t)kv_len * pieces;
  if (idx >= total) return;
  const int tok = (int)(idx / pieces);
  const int byte = (int)(idx % pieces) * 16;
  const int head = byte / a.head_bytes;
  const int inner = byte % a.head_bytes;
  const int32_t* pages = a.pt.page_indices + (a.pt.cu_kv_lens ? (a.pt.cu_kv_lens[a.seq] / a.pt.page_size)
                                                              : (int64_t)a.seq * a.pt.pages_per_seq);
  const int slot = tok / a.pt.page_size;
  const int64_t off = (int64_t)pages[slot] * a.kv.page_stride +
                      (int64_t)(tok - slot * a.pt.page_size) * a.kv.tok_stride +
                      (int64_t)head * a.kv.head_stride + inner;
  st16((char*)a.k_out + (int64_t)tok * a.row_bytes + byte, ld16(a.kv.k_base + off));
  st16((char*)a.v_out + (int64_t)tok * a.row_bytes + byte, ld16(a.kv.v_base + off));
}

// New-token cache write: token j of sequence i lands at position kv_len-q_len+j.
// grid.x covers (token, 16-byte piece); the sequence of a token is found by
// binary search in cu_q_lens.
__global__ __launch_bounds__(256) void rpa_kv_write_kernel(const KvWriteArgs a_in) {
  KvWriteArgs a = a_in;
  if (a.dist) a.num_seqs = min(a.num_seqs, a.dist[2]);
  if (a.dist && a.skip_decode_rows) a.seq_begin = min(a.num_seqs, a.dist[0]);
  if (a.seq_begin >= a.num_seqs) return;  // (no chunk in the bucket: no lengths to wait for, 3.7 -> 1.6 us)
  const int pieces = a.Hkv * a.head_bytes / 16;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int total_tokens = min(a.num_tokens, a.pt.cu_q_lens[a.num_seqs]);
  const int t = (int)(idx / pieces) + (a.seq_begin > 0 ? a.pt.cu_q_lens[a.seq_begin] : 0);
  if (t >= total_tokens) return;
  const int byte = (int)(idx % pieces) * 16;
  int lo = 0, hi = a.num_seqs;  // last i with cu_q_lens[i] <= t
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (a.pt.cu_q_lens[mid] <= t) lo = mid; else hi = mid;
  }
  const int seq = lo;
  const int q0 = a.pt.cu_q_lens[seq], q1 = a.pt.cu_q_lens[seq + 1];
  const int pos = a.pt.kv_lens[seq] - (q1 - q0) + (t - q0);
  if (pos < 0) return;
  const int32_t* pages = a.pt.page_indices + (a.pt.cu_kv_lens ? (a.pt.cu_kv_lens[seq] / a.pt.page_size)
                                                              : (int64_t)seq * a.pt.pages_per_seq);
  const int slot = pos / a.pt.page_size;
  const int head = byte / a.head_bytes;
  const int inner = byte % a.head_bytes;
  const int64_t off = (int64_t)pages[slot] * a.kv.page_stride +
                      (int64_t)(pos - slot * a.pt.page_size) * a.kv.tok_stride +
                      (int64_t)head * a.kv.head_stride + inner;
  const int64_t src = ((int64_t)t * a.Hkv + head) * a.src_head_bytes + inner;
  const bool real = inner < a.src_head_bytes;  // (a narrow head's row ends in zeros)
  st16(const_cast<char*>(a.kv.k_base) + off, real ? ld16(a.keys + src) : u32x4_t{0u, 0u, 0u, 0u});
  st16(const_cast<char*>(a.kv.v_base) + off, real ? ld16(a.values + src) : u32x4_t{0u, 0u, 0u, 0u});
}

// The merge behind the fixed plan's pieces.
template <int HD>
void launch_combine(const DecodeArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)a.Hq * (unsigned)a.num_rows);
#define RPA_COMBINE(SIZE) hipLaunchKernelGGL((rpa_combine_kernel<HD, SIZE>), grid, dim3(merge_threads(SIZE)), 0, st, a)
  switch (merge_size(a, a.num_rows, a.max_splits, a.max_splits)) {
    case kMergeEight: RPA_COMBINE(kMergeEight); break;
    case kMergeSixteen: RPA_COMBINE(kMergeSixteen); break;
    case kMergeAny: RPA_COMBINE(kMergeAny); break;
    default: RPA_COMBINE(kMergeWide); break;
  }
#undef RPA_COMBINE
}

template <bool FP8, Pages PG, bool CAP>
void launch_decode_variant(const DecodeArgs& a, dim3 grid, dim3 block, hipStream_t st) {
  // LDS nobody uses keeps four waves on a CU, one per SIMD: without it the dispatcher doubles workgroups up on some CUs
  // while others stand idle, and a CU draws about 39 bytes per ns at most (fixed plan, 128 rows of 256..2048 tokens x 2
  // heads 47.7 -> 35.6 us; balanced, 56 rows of 512..4096 x 8 heads 99.3 -> 98.3).  Not for grids of many rounds, whose
  // workgroups' starts have to overlap.
  const bool one_round = (int64_t)grid.x * grid.z * (block.x / 64) <= 2048;
  const int forced = tuning().decode_lds_kb;
  const unsigned lds = forced >= 0 ? (unsigned)forced << 10 : !one_round ? 0u : block.x >= 256 ? 84u << 10 : block.x >= 128 ? 54u << 10 : 34u << 10;
  if (a.group_rows) {
    // (one workgroup per CU, too)
    const unsigned parts = std::max(84u << 10, (unsigned)(kRowWaves * min(a.G, 16) * kRowPitch * sizeof(float)));
    if constexpr (!FP8) {
      if (a.q_dim == 64) {
        hipLaunchKernelGGL((rpa_decode_row_kernel<false, PG, CAP, true>), grid, block, parts, st, a);
        return;
      }
    }
    hipLaunchKernelGGL((rpa_decode_row_kernel<FP8, PG, CAP>), grid, block, parts, st, a);
    return;
  }
  // heads of 64 dims (rows of 128, the second half zero): half the bytes.  (Not with the opt-in merge inside the kernel.)
  if constexpr (!FP8) {
    if (a.q_dim == 64 && !(a.balanced && a.merge_counters)) {
      if (!a.balanced) hipLaunchKernelGGL((rpa_decode_splitkv_kernel<1, false, PG, CAP, true>), grid, block, lds, st, a);
      else if constexpr (PG == kHalves) hipLaunchKernelGGL((rpa_decode_balanced_halves_kernel<1, false, CAP, false, true>), grid, block, lds, st, a);
      else hipLaunchKernelGGL((rpa_decode_balanced_kernel<1, false, PG == kBlocks, CAP, false, true>), grid, block, lds, st, a);
      return;
    }
  }
  // (with merge_counters set launch_decode() leaves the merge launch out: the kernel has to merge)
  if (!a.balanced) {
    hipLaunchKernelGGL((rpa_decode_splitkv_kernel<1, FP8, PG, CAP>), grid, block, lds, st, a);
  } else if constexpr (PG == kHalves) {
    if (a.merge_counters) hipLaunchKernelGGL((rpa_decode_balanced_halves_kernel<1, FP8, CAP, true>), grid, block, lds, st, a);
    else hipLaunchKernelGGL((rpa_decode_balanced_halves_kernel<1, FP8, CAP, false>), grid, block, lds, st, a);
  } else if (a.merge_counters) {
    hipLaunchKernelGGL((rpa_decode_balanced_kernel<1, FP8, PG == kBlocks, CAP, true>), grid, block, lds, st, a);
  } else {
    hipLaunchKernelGGL((rpa_decode_balanced_kernel<1, FP8, PG == kBlocks, CAP, false>), grid, block, lds, st, a);
  }
}

template <bool FP8, Pages PG>
void launch_decode_pages(const DecodeArgs& a, dim3 grid, dim3 block, hipStream_t st) {
  // soft cap and logit rounding share the general score path
  if (a.sm.soft_cap != 0.f || a.sm.round_logits != 0) launch_decode_variant<FP8, PG, true>(a, grid, block, st);
  else launch_decode_variant<FP8, PG, false>(a, grid, block, st);
}

hipError_t launch_decode_mt(const DecodeArgs& a, dim3 grid, dim3 block, hipStream_t st) {
  switch (pages_of(a.pt.page_size) * 2 + (a.fp8 ? 1 : 0)) {
    case kLanes * 2: launch_decode_pages<false, kLanes>(a, grid, block, st); break;
    case kLanes * 2 + 1: launch_decode_pages<true, kLanes>(a, grid, block, st); break;
    case kHalves * 2: launch_decode_pages<false, kHalves>(a, grid, block, st); break;
    case kHalves * 2 + 1: launch_decode_pages<true, kHalves>(a, grid, block, st); break;
    case kBlocks * 2: launch_decode_pages<false, kBlocks>(a, grid, block, st); break;
    default: launch_decode_pages<true, kBlocks>(a, grid, block, st); break;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_decode(const DecodeArgs& a, hipStream_t stream) {
  if (a.num_rows <= 0) return hipSuccess;
  const int nw = min(max(a.waves_per_wg, 1), min(4, a.Hkv));  // kv heads walked together by one workgroup
  const int head_groups = (a.Hkv + nw - 1) / nw;
  // more than 16 query heads per kv head: further groups of 16 re-walk the KV (rare: MQA-like shapes)
  const int row_groups = (a.G + 15) / 16;
  if (a.balanced) {
    hipError_t e = launch_decode_mt(a, dim3(a.num_wgs), dim3(a.waves_per_wg * 64), stream);
    if (e != hipSuccess) return e;
    if (!a.merge_counters) {
      const dim3 grid((unsigned)a.Hq * (unsigned)a.num_rows);
      const int64_t pieces = a.num_wgs / std::max<int64_t>(1, (int64_t)a.num_rows * head_groups * row_groups);
      if (merge_size(a, a.num_rows, pieces, a.num_wgs) == kMergeWide)
        hipLaunchKernelGGL((rpa_combine_balanced_kernel<kMergeWide>), grid, dim3(merge_threads(kMergeWide)), 0, stream, a);
      else
        hipLaunchKernelGGL((rpa_combine_balanced_kernel<kMergeAny>), grid, dim3(merge_threads(kMergeAny)), 0, stream, a);
    }
    return hipGetLastError();
  }
  if ((int64_t)a.max_splits * a.num_rows > 0x7fffffffLL || (int64_t)a.Hq * a.num_rows > 0x7fffffffLL)
    return hipErrorInvalidValue;
  dim3 grid((unsigned)max(a.max_splits, 1) * (unsigned)a.num_rows, 1, (a.group_rows ? a.Hkv : head_groups) * row_groups);
  dim3 block(a.group_rows ? kRowWaves * 64 : nw * 64);
  hipError_t e = launch_decode_mt(a, grid, block, stream);
  if (e != hipSuccess) return e;
  if (a.max_splits > 1) {
    launch_combine<128>(a, stream);
    e = hipGetLastError();
  }
  return e;
}

// A few KB of host words as kernel arguments: the words ride in the packet's argument buffer and the store is one more
// kernel of the stream, where a copy is a hand-over to a copy engine and back (five small copies of a step's metadata took
// 20 us of host time and 4 us of the GPU's each).  Up to three launches; beyond, a copy costs less (host memory that is not
// pinned is staged before the call returns).
namespace {
constexpr int kUploadWords = 896;  // 3.5 KB: under the 4 KB that arguments may take
struct UploadWords {
  int32_t w[kUploadWords];
};
__global__ __launch_bounds__(256) void rpa_upload_kernel(int32_t* dst, int n, const UploadWords words) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = words.w[i];
}
}  // namespace

hipError_t launch_upload(int32_t* dst, const int32_t* src, int n, hipStream_t stream) {
  if (n > 3 * kUploadWords) {
    // (not into a graph: a replay would read the host memory again, and the caller may have let go of it)
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    const hipError_t e = hipStreamIsCapturing(stream, &capture);
    if (e != hipSuccess) return e;
    if (capture == hipStreamCaptureStatusNone)
      return hipMemcpyAsync(dst, src, (size_t)n * sizeof(int32_t), hipMemcpyHostToDevice, stream);
  }
  UploadWords words;
  for (int at = 0; at < n; at += kUploadWords) {
    const int m = min(n - at, kUploadWords);
    memcpy(words.w, src + at, (size_t)m * sizeof(int32_t));
    hipLaunchKernelGGL(rpa_upload_kernel, dim3((m + 255) / 256), dim3(256), 0, stream, dst + at, m, words);
  }
  return hipGetLastError();
}

hipError_t launch_gather(const GatherArgs& a, hipStream_t stream) {
  if (a.max_tokens <= 0) return hipSuccess;
  const int64_t total = (int64_t)a.max_tokens * (a.row_bytes / 16);
  const int blocks = (int)((total + 255) / 256);
  hipLaunchKernelGGL(rpa_gather_kernel, dim3(blocks), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_rows256(const DecodeArgs& a, int seq_begin, int seq_end, int max_token_rows, int dist_role,
                          hipStream_t stream) {
  if (seq_end <= seq_begin || max_token_rows <= 0) return hipSuccess;
  if (a.Hkv > 65535) return hipErrorInvalidValue;  // grid.y
  const int nsplit = a.max_splits > 1 ? a.max_splits : 1;
  if ((int64_t)max_token_rows * nsplit > 0x7fffffffLL) return hipErrorInvalidValue;
  const dim3 grid(max_token_rows * nsplit, a.Hkv, (a.G + 15) / 16), block(64);
#define RPA_ROWS256(FP8, PG) hipLaunchKernelGGL((rpa_rows256_kernel<FP8, PG>), grid, block, 0, stream, a, seq_begin, seq_end, dist_role)
  switch (pages_of(a.pt.page_size) * 2 + (a.fp8 ? 1 : 0)) {
    case kLanes * 2: RPA_ROWS256(false, kLanes); break;
    case kLanes * 2 + 1: RPA_ROWS256(true, kLanes); break;
    case kHalves * 2: RPA_ROWS256(false, kHalves); break;
    case kHalves * 2 + 1: RPA_ROWS256(true, kHalves); break;
    case kBlocks * 2: RPA_ROWS256(false, kBlocks); break;
    default: RPA_ROWS256(true, kBlocks); break;
  }
#undef RPA_ROWS256
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || nsplit == 1) return e;
  if ((int64_t)a.Hq * a.num_rows > 0x7fffffffLL) return hipErrorInvalidValue;
  launch_combine<256>(a, stream);
  return hipGetLastError();
}

hipError_t launch_kv_write(const KvWriteArgs& a, hipStream_t stream) {
  if (a.num_tokens <= 0 || a.num_seqs <= a.seq_begin) return hipSuccess;
  const int64_t total = (int64_t)(a.num_tokens - a.seq_begin) * (a.Hkv * a.head_bytes / 16);
  const int blocks = (int)((total + 255) / 256);
  hipLaunchKernelGGL(rpa_kv_write_kernel, dim3(blocks), dim3(256), 0, stream, a);
  return hipGetLastError();
}

}  // namespace rpa
