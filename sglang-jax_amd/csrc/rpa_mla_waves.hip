// Absorbed-MLA decode rows on gfx950, a wave per tile: 16 heads per workgroup.
//
// The kernels of rpa_mla.hip are made for 128 heads that share a row of latents.  Where a call has 16 heads (a tensor-parallel share), or so few
// rows that its workgroups leave most of the chip idle, the matrix work is little and what costs is the chain of a step: barriers, partial
// scores exchanged through LDS, one wave's operands behind another's.  Here the four waves of a workgroup, one per SIMD, take the tiles of a piece
// in turn, and each has everything of its tile to itself: the copies into its own part of LDS, the scores over all 576 dims, the softmax, the
// second product into all 512 dims.  No barrier between tiles; the waves' results meet in LDS at the end of the piece.
//   tile              16 tokens (bf16) or 32 (e4m3): 18 KB either way, two per wave on their way or in use
//   S^T[tok, head]    18 MFMA 16x16x32 per 16 tokens; A = rows by ds_read_b128, B = Q^T in registers
//   O^T[dim, head]    32 MFMA, 16x16x16 on 16 tokens, 16x16x32 on 32; A = V^T by the transposing reads of 16- or 8-bit elements
//   e4m3              stays as it is in LDS and is widened in registers, two elements an instruction (exact)
// More than 16 heads are siblings: workgroups of their own over the same tokens, side by side on one XCD, whose L2 the tiles come from.
//
// What bounds it: 64 rows of 2047..16383 bf16 tokens x 16 heads read 5.3 TB/s (112 us; 128 with tiles shared by the waves, rpa_mla.hip), where the
// same bytes alone take 96; e4m3 119 -> 79, there the instructions of a lone wave per SIMD do (0.55 us per 32 tokens and workgroup, from L2).
// Small calls are a chain: one row of 500 tokens in eight pieces, us: arguments 0.5, lengths 0.6, page ids 0.8, queries and tiles 2, a tile 1.2, the waves'
// merge 1.7, rows out 0.8; 13.3 -> 12.0 with the launches for 16 heads, 17.6 -> 12.3 for 64, 20.4 -> 13.0 for 128.
//
// All 512 registers of a lane are taken.  e4m3 rows spill 18 (balanced) or 4 (fixed pieces) more, 76 or 20 bytes of scratch: what the loop over
// tiles does not touch, written before it and read behind it.  bf16 rows spill none.
//
// A row of a tile has a copy instruction of its own (e4m3: two rows), so pages of any size, the row's last token in place of those past its
// end and the new token out of the caller's rows are a matter of addresses; tiles that lie in one page have one address for all.

#include "rpa_common.h"
#include "rpa_dsa.h"
#include "rpa_kernels.h"
#include "rpa_mla_common.h"

namespace rpa {
namespace {

constexpr int kWaves = 4;
constexpr int kLineB = 1056;                  // 1024 bytes of kv_c (one bf16 row, two e4m3 rows) and 32 of padding: 16 rows in 8 places
constexpr int kLines = 16;
constexpr int kRopeAt = kLines * kLineB;      // k_pe of the tile's rows, chunks of 16 bytes swizzled
constexpr int kTileB = kRopeAt + 2048;
constexpr int kRingB = kWaves * 2 * kTileB;
constexpr int kCopies = kLines + 2;           // copy instructions of a tile
constexpr int kIds = 4;                       // tiles whose page ids are in LDS

typedef __attribute__((address_space(3))) int32_t* lds_ids_t;

__device__ __forceinline__ f32x4_t mfma16_k16(u32x2_t a, u32x2_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4_t, a), __builtin_bit_cast(s16x4_t, b), c, 0, 0, 0);
}

// Lane r of 16: byte (r & 1) * 8 of eight rows' 16 at p, row r >> 1; comes back with byte r of the eight rows.
__device__ __forceinline__ u32x2_t lds_tr8(const char* p) {
  typedef int i32x2_t __attribute__((ext_vector_type(2)));
  typedef __attribute__((address_space(3))) i32x2_t* lds_ptr_t;
  return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_ptr_t)(p)));
}

__device__ __forceinline__ u32x4_t widen(uint32_t w0, uint32_t w1) {
  const u32x2_t lo = fp8x4_to_bf16x4(w0), hi = fp8x4_to_bf16x4(w1);
  return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
}

__device__ __forceinline__ uint64_t lane_of(uint64_t x, int lane) {
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)x, lane), hi = __builtin_amdgcn_readlane((uint32_t)(x >> 32), lane);
  return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t from_lane(uint64_t x, int lane) {
  const uint32_t lo = __builtin_amdgcn_ds_bpermute(lane * 4, (int)(uint32_t)x), hi = __builtin_amdgcn_ds_bpermute(lane * 4, (int)(uint32_t)(x >> 32));
  return ((uint64_t)hi << 32) | lo;
}

// f(0), f(1), .. f(N - 1), each number a type
template <int N, int I = 0, class F>
__device__ __forceinline__ void each(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    each<N, I + 1>(f);
  }
}

// Copy number `i` of a tile whose rows have one address: to LDS at dst + at_lds, from `base` + at + step.  s_nop: a scalar that a vector instruction
// wrote may be an address five wait states later (m0 one: the addition).
template <bool NT, bool FIRST>
__device__ __forceinline__ void copy_line(uint32_t dst, int at_lds, uint64_t base, uint32_t& at, uint32_t step) {
#define RPA_LINE(WAIT, POLICY)                                                                                                          \
  asm volatile(WAIT "s_add_u32 m0, %[dst], %[lds]\n\tv_add_u32 %[at], %[step], %[at]\n\tglobal_load_lds_dwordx4 %[at], %[base]" POLICY \
               : [at] "+v"(at) : [dst] "s"(dst), [lds] "i"(at_lds), [base] "s"(base), [step] "s"(step) : "memory", "m0", "scc")
  if constexpr (FIRST && NT) RPA_LINE("s_nop 4\n\t", " nt");
  else if constexpr (FIRST) RPA_LINE("s_nop 4\n\t", "");
  else if constexpr (NT) RPA_LINE("", " nt");
  else RPA_LINE("", "");
#undef RPA_LINE
}

// One workgroup, one row, 16 heads from head_base on, tokens [t_begin, t_end).  Tokens from new_begin on are rows new_row .. of the caller's
// new_kv_c / new_k_pe (a row's newest token; none: new_begin = kv_len); put: they also go into the cache, from the tile that has them.
// ids: first_ids holds the first 64 pages' ids, a lane each.  NT: what no other workgroup reads leaves the caches first (64 ragged rows x 16
// heads 136 -> 114 us).
template <bool FP8, bool NT>
__device__ __forceinline__ void mla_segment_waves(const MlaDecodeArgs& a, const MlaRow mr, int head_base, int t_lo, int t_begin, int t_end,
                                                  const MlaDest dest, char* ring, const char* new_kv_c, const char* new_k_pe, int new_begin,
                                                  int new_row, bool put, bool ids, int first_ids) {
  constexpr int kTile = FP8 ? 32 : 16;   // tokens
  constexpr int kHalves = kTile / 16;
  constexpr int kEs = FP8 ? 1 : 2;       // bytes per element
  __shared__ int32_t id_ring[kWaves][kIds][64];
  __shared__ float refs[kWaves][2][16];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int kv_len = mr.kv_len, last_tok = kv_len - 1;
  const int P = a.pt.page_size, shift = (P & (P - 1)) == 0 ? 31 - __builtin_clz(P) : -1;
  const int32_t* pages = a.pt.page_indices + (a.pt.cu_kv_lens ? (int64_t)(scalar_load_i32(a.pt.cu_kv_lens + mr.seq) / P)
                                                             : (int64_t)mr.seq * a.pt.pages_per_seq);
  const int row_bytes = a.row_stride * kEs;
  const int64_t page_stride = (int64_t)row_bytes * P;
  const int rope_byte = a.rope_offset * kEs;
  auto slot_of = [&](int tok) { return shift >= 0 ? tok >> shift : tok / P; };
  const int first_slot = slot_of(t_begin);  // (of first_ids)
  if (!FP8 && t_lo - t_begin >= 16) t_begin += 16;  // (pieces begin at a multiple of 32)
  char* const mine = ring + wave * 2 * kTileB;
  const uint32_t mine_lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)mine);
  const int n = max(0, ((t_end - t_begin + kTile - 1) / kTile - wave + kWaves - 1) / kWaves);  // this wave's tiles
  auto begin_of = [&](int k) { return t_begin + (wave + k * kWaves) * kTile; };
  auto row_of = [&](int k) { return min(begin_of(k) + (lane & (kTile - 1)), last_tok); };  // the token of the lane's row
  const bool ids_here = ids && slot_of(t_end - 1) - first_slot < 64;
  auto id_in_register = [&](int k) { return __builtin_amdgcn_ds_bpermute((slot_of(row_of(k)) - first_slot) * 4, first_ids); };

  // ---- page ids of the first two tiles and the queries, in one round trip.  Column c = head head_base + c; bf16: k-step ks has dims 32 ks + 8 g ..;
  // e4m3: a read of 16 bytes is two steps, dims 64 (ks / 2) + 16 g + 8 (ks & 1) ..
  // (An id from a register brings its copies at once, and the queries follow them; behind the queries it would wait for these.)
  typedef const __attribute__((address_space(1))) int32_t* global_i32_t;  // (where the table was written by this kernel the compiler does not know it)
  int id0 = 0, id1 = 0;
  u32x4_t qB[18];
  auto load_queries = [&]() __attribute__((always_inline)) {
    const int head = min(head_base + c, a.Hq - 1);
    const uint16_t* qn = a.ql_nope + ((int64_t)mr.tq * a.Hq + head) * 512 + g * (FP8 ? 16 : 8);
    const uint16_t* qr = a.q_pe + ((int64_t)mr.tq * a.Hq + head) * 64 + g * (FP8 ? 16 : 8);
#pragma unroll
    for (int ks = 0; ks < 18; ++ks) {
      const int d = FP8 ? (ks >> 1) * 64 + (ks & 1) * 8 : ks * 32;
      qB[ks] = ld16(ks < 16 ? qn + d : qr + (d - 512));
    }
  };
  if (ids_here) {
    id0 = id_in_register(0);
    id1 = id_in_register(1);
  } else {
    id0 = ((global_i32_t)pages)[slot_of(row_of(0))];
    id1 = ((global_i32_t)pages)[slot_of(row_of(1))];
    load_queries();
    asm volatile("" : "+v"(id0), "+v"(id1));
  }

  // ---- a tile's copies
  // the lane's offsets from the base of 16 rows, a step short: a line (e4m3: of two rows), k_pe
  const uint32_t step = (FP8 ? 2 : 1) * row_bytes;
  const uint32_t line_at = (FP8 ? (lane >> 5) * row_bytes + (lane & 31) * 16 : lane * 16) - step;
  const uint32_t pe_at = (FP8 ? (lane >> 2) * row_bytes + rope_byte + ((lane ^ (lane >> 4)) & 3) * 16
                              : (lane >> 3) * row_bytes + rope_byte + ((lane ^ (lane >> 4)) & 7) * 16) - step;
  const uint32_t pe_at2 = FP8 ? pe_at : (8 + (lane >> 3)) * row_bytes + rope_byte + ((lane ^ (4 + (lane >> 4))) & 7) * 16 - step;
  uint64_t put_at = 0;  // where the new token of the tile asked for last belongs
  auto ask_ids = [&](int k) __attribute__((always_inline)) {  // two tiles ahead of the rows: landed whenever the tile in between is waited for
    if (ids_here || k >= n) return;
    const uint32_t m0v = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ids_t)&id_ring[wave][k & (kIds - 1)][0]);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(m0v), "v"(pages + slot_of(row_of(k))) : "memory", "m0");
  };
  // pages of whole 16 rows, every row of the tile in the cache: one address per 16 rows
  auto plain = [&](int k) { return P % 16 == 0 && begin_of(k) + kTile <= min(kv_len, new_begin); };
  auto half_at = [&](int k, int h, int id) {
    const int pg = __builtin_amdgcn_readlane(id, 16 * h), t = begin_of(k) + 16 * h;
    return reinterpret_cast<uint64_t>((pg < 0 ? a.extra_rows : a.cache) + (int64_t)(pg < 0 ? ~pg : pg) * page_stride + (int64_t)(t - slot_of(t) * P) * row_bytes);
  };
  auto copy_plain = [&](auto number, uint32_t dst, uint64_t lo, uint64_t hi, uint32_t& at, uint32_t& pe, uint32_t& pe2) __attribute__((always_inline)) {
    constexpr int i = decltype(number)::value;
    if (FP8 && i == 8) at = line_at;
    if constexpr (i < kLines) copy_line<NT, i == 0>(dst, i * kLineB, i < 8 ? lo : hi, at, step);
    else if constexpr (i == kLines) copy_line<NT, false>(dst, kRopeAt, lo, pe, step);
    else copy_line<NT, false>(dst, kRopeAt + 1024, hi, pe2, step);
  };
  // others row by row: lane r works out where row r is
  auto copy_rows = [&](int k, int id) __attribute__((always_inline)) {
    char* dst = mine + (k & 1) * kTileB;
    const int tok = row_of(k);
    const char* in_cache = (id < 0 ? a.extra_rows : a.cache) + (int64_t)(id < 0 ? ~id : id) * page_stride + (int64_t)(tok - slot_of(tok) * P) * row_bytes;
    const bool is_new = tok >= new_begin;
    const int64_t from = new_row + tok - new_begin;
    const uint64_t kv = reinterpret_cast<uint64_t>(is_new ? new_kv_c + from * (512 * kEs) : in_cache);
    const uint64_t pe = reinterpret_cast<uint64_t>(is_new ? new_k_pe + from * (64 * kEs) : in_cache + rope_byte);
    if (put && begin_of(k) + kTile > new_begin) put_at = lane_of(reinterpret_cast<uint64_t>(in_cache), new_begin - begin_of(k));
#pragma unroll
    for (int i = 0; i < kLines; ++i) {
      if constexpr (FP8) async_copy16(reinterpret_cast<const char*>(from_lane(kv, 2 * i + (lane >> 5))) + (lane & 31) * 16, dst + i * kLineB);
      else async_copy16(reinterpret_cast<const char*>(lane_of(kv, i)) + lane * 16, dst + i * kLineB);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if constexpr (FP8) async_copy16(reinterpret_cast<const char*>(from_lane(pe, 16 * h + (lane >> 2))) + ((lane ^ (lane >> 4)) & 3) * 16, dst + kRopeAt + h * 1024);
      else async_copy16(reinterpret_cast<const char*>(from_lane(pe, 8 * h + (lane >> 3))) + ((lane ^ (4 * h + (lane >> 4))) & 7) * 16, dst + kRopeAt + h * 1024);
    }
  };
  auto ask = [&](int k, int id) __attribute__((always_inline)) {
    ask_ids(k + 2);
    if (plain(k)) {
      const uint64_t lo = half_at(k, 0, id), hi = FP8 ? half_at(k, 1, id) : lo;
      uint32_t at = line_at, pe = pe_at, pe2 = pe_at2;
      const uint32_t dst = mine_lds + (k & 1) * kTileB;
      each<kCopies>([&](auto i) __attribute__((always_inline)) { copy_plain(i, dst, lo, hi, at, pe, pe2); });
    } else {
      copy_rows(k, id);
    }
  };
  // The compiler counts no copies: what it waits for next, the queries, is everything in flight, two tiles among it.
  if (n > 0) ask(0, id0);
  if (n > 1) ask(1, id1);
  if (ids_here) load_queries();
  // (zeros where they belong, in the accumulation registers, while the copies are on their way: through the vector registers and behind the wait
  // they were 0.8 us of a piece)
  f32x4_t acc[32];
#pragma unroll
  for (int j = 0; j < 32; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float zero;
      asm volatile("v_accvgpr_write_b32 %0, 0" : "=a"(zero));
      acc[j][e] = zero;
    }
#pragma unroll
  for (int ks = 0; ks < 18; ++ks) asm volatile("" : "+v"(qB[ks]));

  const float scale2 = a.sm.sm_scale * kLog2e;
  const float mask2 = fmaxf(a.sm.mask_value * kLog2e, -3.0e38f);
  float m = -INFINITY, l = 0.f, raise = 0.f;
  // LDS places of the lane inside a tile
  const int k_off = FP8 ? (c >> 1) * kLineB + (c & 1) * 512 + g * 16 : c * kLineB + g * 16;
  const int vr = c >> 1;  // e4m3: the lane's row of eight
  const int v_tok = FP8 ? (vr < 4 ? 4 * g + vr : 12 + 4 * g + vr) : 4 * g + (c >> 2);
  const int v_off = FP8 ? (v_tok >> 1) * kLineB + (v_tok & 1) * 512 + (c & 1) * 8 : v_tok * kLineB + (c & 3) * 8;
  auto rope_off = [&](int b, int chunk) { return kRopeAt + (FP8 ? (16 * b + c) * 64 + ((chunk ^ (c >> 2)) & 3) * 16 : c * 128 + ((chunk ^ (c >> 1)) & 7) * 16); };

  // The reference of the probabilities is the first tile's maximum, and follows only a maximum 2^60 above it: f32 sums have the room, and
  // bf16 rounds a probability of any size by the same part of it.  The sum is that of the rounded probabilities and a piece leaves its row
  // divided by it, so that where a few tokens are all of a row their rounding cancels.  The loop is left for the accumulators to move.
  int k = 0;
  for (;;) {
    for (; k < n; ++k) {
      // this tile has landed once no more than the next one's copies are on their way
      if (k + 1 < n) __builtin_amdgcn_s_waitcnt(0x0F70 | (kCopies & 15) | ((kCopies >> 4) << 14));
      else __builtin_amdgcn_s_waitcnt(0x0F70);
      asm volatile("" ::: "memory");
      const char* tile = mine + (k & 1) * kTileB;
      const int tb = begin_of(k);
      // ---- everything that is read from the tile, at once: its place is free again behind the softmax
      u32x4_t kx[18];
      u32x2_t vx[32];
#pragma unroll
      for (int i = 0; i < 18; ++i) {
        if constexpr (FP8) kx[i] = lds_ld16(tile + (i < 16 ? k_off + (i & 1) * 8 * kLineB + (i >> 1) * 64 : rope_off(i & 1, g)));
        else kx[i] = lds_ld16(tile + (i < 16 ? k_off + i * 64 : rope_off(0, (i - 16) * 4 + g)));
      }
      const int id = k + 2 < n ? ids_here ? id_in_register(k + 2) : id_ring[wave][(k + 2) & (kIds - 1)][lane] : 0;
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        if constexpr (FP8) vx[j] = lds_tr8(tile + v_off + j * 16);
        else vx[j] = lds_tr16(tile + v_off + j * 32);
      }
      __builtin_amdgcn_sched_barrier(0);
      // ---- scores
      f32x4_t s[kHalves][2];
#pragma unroll
      for (int b = 0; b < kHalves; ++b) s[b][0] = s[b][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 18; ++i) {
        if constexpr (FP8) {
          s[i & 1][0] = mfma16(widen(kx[i][0], kx[i][1]), qB[i & ~1], s[i & 1][0]);
          s[i & 1][1] = mfma16(widen(kx[i][2], kx[i][3]), qB[i | 1], s[i & 1][1]);
        } else {
          s[0][i & 1] = mfma16(kx[i], qB[i], s[0][i & 1]);
        }
      }
      // ---- probabilities
      float x[4 * kHalves];
#pragma unroll
      for (int i = 0; i < 4 * kHalves; ++i) x[i] = (s[i >> 2][0][i & 3] + s[i >> 2][1][i & 3]) * scale2;
      if (tb + kTile > kv_len || tb < t_lo) {
#pragma unroll
        for (int i = 0; i < 4 * kHalves; ++i) {
          const int tok = tb + 16 * (i >> 2) + 4 * g + (i & 3);
          if (tok >= kv_len || tok < t_lo) x[i] = mask2;
        }
      }
      float mx = x[0];
#pragma unroll
      for (int i = 1; i < 4 * kHalves; ++i) mx = fmaxf(mx, x[i]);
      mx = swap_max(swap16_max(mx));
      if (k == 0) m = fmaxf(mx, -3.0e38f);  // (scores that overflow to -infinity count nothing, also where they are all of a tile)
      raise = mx;
      if (__builtin_amdgcn_ballot_w64(mx > m + 60.0f) != 0) break;
      u32x4_t pB = {0u, 0u, 0u, 0u}, pR = {0u, 0u, 0u, 0u};  // rounded, and what rounding left of them
      float whole = 0.f, rest = 0.f;
#pragma unroll
      for (int i = 0; i < 2 * kHalves; ++i) {
        const float p0 = fast_exp2(x[2 * i] - m), p1 = fast_exp2(x[2 * i + 1] - m);
        pB[i] = pack_bf16x2(p0, p1);
        const float h0 = bf16_lo_to_f32(pB[i]), h1 = bf16_hi_to_f32(pB[i]);
        pR[i] = pack_bf16x2(p0 - h0, p1 - h1);
        whole += h0 + h1;
        rest += bf16_lo_to_f32(pR[i]) + bf16_hi_to_f32(pR[i]);
      }
      // bf16: the remainders are the other half of a 16x16x32's operand.  e4m3: a second product, where some head's tile is a large part of its row.
      const bool exact = !FP8 || __builtin_amdgcn_ballot_w64(whole > 0.125f * l) != 0;
      l += exact ? whole + rest : whole;
      // ---- the new token into the cache
      if (put && tb + kTile > new_begin) {
        const int r = new_begin - tb;
        char* row = reinterpret_cast<char*>(put_at);
        if constexpr (FP8) {
          const int t = min(lane, 35);
          const u32x4_t y = lds_ld16(tile + (t < 32 ? (r >> 1) * kLineB + (r & 1) * 512 + t * 16 : kRopeAt + r * 64 + (((t - 32) ^ (r >> 2)) & 3) * 16));
          if (lane < 36) st16(row + (t < 32 ? t * 16 : rope_byte + (t - 32) * 16), y);
        } else {
          const u32x4_t y = lds_ld16(tile + r * kLineB + lane * 16), z = lds_ld16(tile + kRopeAt + r * 128 + ((lane ^ (r >> 1)) & 7) * 16);
          st16(row + lane * 16, y);
          if (lane < 8) st16(row + rope_byte + lane * 16, z);
        }
      }
      // ---- the copies of the tile after next, then the second product
      __builtin_amdgcn_s_waitcnt(0xC07F);  // (lgkmcnt(0): every read is back)
      asm volatile("" ::: "memory");
      if (k + 2 < n) ask(k + 2, id);
      if constexpr (FP8) {
#pragma unroll 1
        for (int pass = exact ? 2 : 1; pass > 0; --pass) {  // (a loop: behind a branch the accumulators would be there twice)
          const u32x4_t p = pass == 2 ? pR : pB;
#pragma unroll
          for (int j = 0; j < 32; ++j) acc[j] = mfma16(widen(vx[j][0], vx[j][1]), p, acc[j]);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 32; ++j) acc[j] = mfma16(u32x4_t{vx[j][0], vx[j][1], vx[j][0], vx[j][1]}, u32x4_t{pB[0], pB[1], pR[0], pR[1]}, acc[j]);
      }
    }
    if (k >= n) break;
    const float m_new = fmaxf(m, raise), alpha = fast_exp2(m - m_new);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int j = 0; j < 32; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float x = acc[j][e], t;  // (in place: through vector registers it would be there in every tile)
        asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\tv_accvgpr_write_b32 %0, %1" : "+a"(x), "=&v"(t) : "v"(alpha));
        acc[j][e] = x;
      }
  }

  // ---- the waves' results meet.  Lane (c, g) holds head head_base + c, dims 16 j + 4 g + r in acc[j][r]; wave w finishes dims 128 w ..
  l = swap_sum(swap16_sum(l));
  if (g == 0) {
    refs[wave][0][c] = m;
    refs[wave][1][c] = l;
  }
  __syncthreads();  // (and every wave has left its tiles)
#pragma unroll
  for (int j = 0; j < 32; ++j) *reinterpret_cast<f32x4_t*>(ring + ((wave * 32 + j) * 64 + lane) * 16) = acc[j];
  float f[kWaves], top = refs[0][0][c], sum = 0.f;
#pragma unroll
  for (int w = 1; w < kWaves; ++w) top = fmaxf(top, refs[w][0][c]);
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    f[w] = fast_exp2(refs[w][0][c] - top);
    sum += refs[w][1][c] * f[w];
  }
  const float inv = dest.final_rows ? a.out_scale / sum : sum == 0.f ? 0.f : 1.0f / sum;  // (a piece of nothing but -infinity weighs nothing)
  __syncthreads();
  f32x4_t own[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) own[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < kWaves; ++w)
#pragma unroll
    for (int i = 0; i < 8; ++i) own[i] += *reinterpret_cast<const f32x4_t*>(ring + ((w * 32 + wave * 8 + i) * 64 + lane) * 16) * (f[w] * inv);
  const int head = head_base + c;
  u32x4_t out[4];
#pragma unroll
  for (int j = 0; j < 8; j += 2)
    out[j / 2] = row_of_16(u32x2_t{pack_bf16x2(own[j][0], own[j][1]), pack_bf16x2(own[j][2], own[j][3])},
                           u32x2_t{pack_bf16x2(own[j + 1][0], own[j + 1][1]), pack_bf16x2(own[j + 1][2], own[j + 1][3])});
  if (head < a.Hq) {
    uint16_t* row = dest.final_rows ? a.out + ((int64_t)mr.tq * a.Hq + head) * 512 : a.ws_o + (dest.base + head) * 512;
#pragma unroll
    for (int j = 0; j < 8; j += 2) st16(row + (wave * 8 + j) * 16 + g * 8, out[j / 2]);
    if (!dest.final_rows && wave == 0 && g == 0) {
      a.ws_ml[(dest.base + head) * 2 + 0] = sum == 0.f ? top : top + __builtin_amdgcn_logf(sum);
      a.ws_ml[(dest.base + head) * 2 + 1] = sum == 0.f ? 0.f : 1.0f;
    }
  }
  __syncthreads();  // (the next piece's copies land where this one's rows met)
}

// The row's newest token, where the call brings it.
struct NewToken {
  int begin, row;
};
// Copies into LDS move aligned chunks of 16 bytes: rows of the caller's that begin elsewhere go through registers into the cache, and come from there.
__device__ __forceinline__ bool in_chunks(const char* kv_c, const char* k_pe) {
  return ((reinterpret_cast<uint64_t>(kv_c) | reinterpret_cast<uint64_t>(k_pe)) & 15) == 0;
}
template <bool FP8>
__device__ __forceinline__ NewToken new_token(const MlaDecodeArgs& a, const MlaRow& mr, int t_end, bool& put) {
  if (!a.new_kv_c) {
    put = false;
    return {mr.kv_len, 0};
  }
  const int q0 = scalar_load_i32(a.pt.cu_q_lens + mr.seq), count = scalar_load_i32(a.pt.cu_q_lens + mr.seq + 1) - q0;
  const bool direct = in_chunks(a.new_kv_c, a.new_k_pe);
  if (!direct) put = t_end > mr.kv_len - count;  // (by every workgroup that reads a new token, the same bytes: each follows its own stores)
  if (!direct || count != 1) {  // (not a decode row: every token in front of everything)
    if (put) {
      put_new_row<FP8>(a, mr.seq, mr.kv_len);
      if (!direct) wait_all_loads();  // (and stores)
      put = false;
    }
  }
  return {direct ? mr.kv_len - count : mr.kv_len, q0};
}

// ---- fixed plan: workgroups (piece, sibling), pieces of a row one after the other.  SPARSE: the rows' page tables are written here first.
template <bool FP8, bool NT, bool SPARSE>
__global__ __launch_bounds__(64 * kWaves, 1) void rpa_mla_waves_kernel(const MlaDecodeArgs a) {
  __shared__ __attribute__((aligned(1024))) char ring[kRingB];
  fetch_arguments<MlaDecodeArgs>();
  const Sibling sib = sibling(a);
  const int nsp = max(a.max_splits, 1);
  int row_id = sib.of / nsp;
  const int split = sib.of - row_id * nsp;
  if (row_id >= a.num_rows) return;
  MlaDest dest;
  dest.final_rows = a.max_splits == 1;
  const int head_base = sib.unit * 16;
  if constexpr (SPARSE) {
    sparse::Piece p = {};
    if (!sparse::begin_piece<64 * kWaves, true>(a, row_id, split, ring, p)) return;
    const MlaRow mr = {row_id, p.kv_len, row_id, true};
    dest.base = ((int64_t)row_id * a.max_splits + split) * a.Hq;
    MlaDecodeArgs b = a;
    // (behind the table's barrier: page ids are read as what nobody writes, and could be asked for in front of it)
    asm volatile("" : "+s"(b.pt.page_indices)::"memory");
    const bool whole_pages = a.sparse.k_pages_max > 0;
    const int new_begin = a.sparse.new_kv_c && in_chunks(a.sparse.new_kv_c, a.sparse.new_k_pe) ? p.kv_len - 1 : p.kv_len;
    mla_segment_waves<FP8, NT>(b, mr, head_base, p.t_lo, p.t_begin, p.t_end, dest, ring, a.sparse.new_kv_c, a.sparse.new_k_pe, new_begin, row_id, false,
                               whole_pages, p.page_ids);
    return;
  }
  if (a.rows_are_tokens) row_id = a.num_rows - 1 - row_id;
  const MlaRow mr = mla_row(a, row_id);
  if (!mr.valid) return;
  const int kv_len = mr.kv_len;
  if (kv_len <= 0) return;
  const int t_lo = (a.sm.window > 0) ? max(0, kv_len - a.sm.window) : 0;
  const int t0 = t_lo & ~(kTok - 1);
  const int t_begin = t0 + split * a.chunk;
  if (t_begin >= kv_len) return;
  const int t_end = (split == a.max_splits - 1) ? kv_len : min(kv_len, t_begin + a.chunk);
  dest.base = ((int64_t)row_id * a.max_splits + split) * a.Hq;
  bool put = sib.unit == 0 && t_end == kv_len;
  const NewToken nt = new_token<FP8>(a, mr, t_end, put);
  mla_segment_waves<FP8, NT>(a, mr, head_base, t_lo, t_begin, t_end, dest, ring, a.new_kv_c, a.new_k_pe, nt.begin, nt.row, put, false, 0);
}

// ---- balanced plan (mla_balanced_body); all heads of a share's rows are its siblings', so the line has one unit per row
template <bool FP8, bool NT>
__global__ __launch_bounds__(64 * kWaves, 1) void rpa_mla_waves_balanced_kernel(const MlaDecodeArgs a) {
  __shared__ __attribute__((aligned(1024))) char ring[kRingB];
  fetch_arguments<MlaDecodeArgs>();
  const int unit = sibling(a).unit;
  mla_balanced_body<FP8, false>(a, [&](const MlaRow& mr, int, int t_lo, int t_begin, int t_end, const MlaDest& dest, int) __attribute__((always_inline)) {
    bool put = unit == 0 && t_end == mr.kv_len;
    const NewToken nt = new_token<FP8>(a, mr, t_end, put);
    mla_segment_waves<FP8, NT>(a, mr, unit * 16, t_lo, t_begin, t_end, dest, ring, a.new_kv_c, a.new_k_pe, nt.begin, nt.row, put, false, 0);
  });
}

template <bool FP8, bool NT>
void launch(const MlaDecodeArgs& a, hipStream_t stream) {
  const int64_t pieces = a.balanced ? a.num_wgs : (int64_t)std::max(a.max_splits, 1) * a.num_rows;
  const dim3 grid((unsigned)(a.siblings > 1 ? (pieces + 7) / 8 * 8 * a.siblings : pieces));
  if (a.balanced) {
    hipLaunchKernelGGL((rpa_mla_waves_balanced_kernel<FP8, NT>), grid, dim3(64 * kWaves), 0, stream, a);
    return;
  }
  if (a.sparse.topk) hipLaunchKernelGGL((rpa_mla_waves_kernel<FP8, NT, true>), grid, dim3(64 * kWaves), 0, stream, a);
  else hipLaunchKernelGGL((rpa_mla_waves_kernel<FP8, NT, false>), grid, dim3(64 * kWaves), 0, stream, a);
}

}  // namespace

hipError_t launch_mla_waves(const MlaDecodeArgs& a, hipStream_t stream) {
  // Rows of sequences and selections of 16 heads are one workgroup's and pass through the caches once (NT of mla_segment_waves).  A chunk's tokens all read
  // the same prefix, out of L2: 116 calls of 40..1000 tokens on up to 8000 x 16 heads, non-temporal -> plain, 1.026 x in the geometric mean, 4 chunks of
  // 86..326 on 441..882 98.7 -> 90.3 us, e4m3 4 of 63..292 on 463 83.6 -> 78.7; what loses most are prefixes larger than an L2, 142 on 6400 137 -> 140.
  const bool alone = a.siblings <= 1 && !a.rows_are_tokens;
  if (a.fp8) alone ? launch<true, true>(a, stream) : launch<true, false>(a, stream);
  else alone ? launch<false, true>(a, stream) : launch<false, false>(a, stream);
  return hipGetLastError();
}

}  // namespace rpa
