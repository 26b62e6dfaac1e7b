// Flash-style prefill / mixed kernel for ragged paged attention on gfx950.
//
// One workgroup (4 waves) owns a tile of 128 query positions of one query head
// of one sequence; wave w owns 32 of them.  KV is walked in tiles of 64 tokens
// gathered through the page table into a two-deep LDS ring (tile t+1 arrives
// while tile t is consumed, one barrier per tile):
//   S^T[tok, q]  = K . Q^T        v_mfma_f32_32x32x16_bf16, A = K rows from LDS,
//                                 B = Q^T held in registers for the whole loop
//   online softmax per query column (in-lane over tokens + one lane swap)
//   O^T[dim, q] += V^T . P^T      A = V^T from LDS, B = P^T straight from the
//                                 S^T result registers
// The S^T result layout (lane = query, registers = tokens) is the B operand
// layout of the second product when the 16 tokens of a k-step are ordered
// 16kk + 8*(i/4) + 4h + i%4 -- no data crosses lanes between the two products.
//
// Two data paths feed the LDS ring:
//   * bf16 cache ("async"): global_load_lds_dwordx4 copies 16-byte chunks straight
//     into LDS, rows kept row-major with XOR-swizzled chunk positions (no padding,
//     no staging registers).  K operands are ds_read_b128; V^T operands come from
//     the row-major V rows through the transposing LDS read ds_read_b64_tr_b16.
//   * fp8 cache ("staged"): rows pass through registers, are dequantised to bf16
//     once, and V is transposed in registers (v_perm_b32) before it is written.
//
// Workgroup ids are remapped so that everything that reads one kv head of one
// sequence runs on the same XCD (same L2) while the ragged sequences are spread
// evenly over the 8 XCDs: hardware deals workgroup n to XCD n % 8.

#include <cstdlib>
#include <type_traits>
#include <utility>

#include "rpa_prefill_common.h"

namespace rpa {

using namespace pf;

namespace {

// f(0), f(1), ... f(N - 1), each with its number as a compile-time constant
template <class F, int... I>
__device__ __forceinline__ void unroll_seq(F f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void unroll_n(F f) {
  unroll_seq(f, std::make_integer_sequence<int, N>{});
}

// A 64-token tile of 128-wide heads: its 32 operand fragments in the order of their use -- K of the scores (f < 16: k-step f >> 1,
// half f & 1), V^T of the second product (half, k-step, dim tile) -- AHEAD of them requested ahead of the matrix instruction
// that takes them, across the softmax in between.  Left to itself the compiler requests a fragment or two and waits for it.
// With the copies' scalar bases (RowFeed), 16-token pages, 32 / 8 heads: 4 chunks of 2048 on 2048 .. 4096 659 -> 553 us, 3639 tokens
// x 64 heads on 5000 929 -> 755, 8 chunks of 64-wide heads 118 -> 94; soft cap, 64-token pages 750 -> 727; e4m3 677 -> 660.
// `request(f, frag)` reads fragment f.  AHEAD = 1: no order of ours (kernels whose options leave no registers for it).
template <int AHEAD, class Request>
__device__ __forceinline__ void tile_scores(f32x16_t (&S)[2], u32x4_t (&frag)[AHEAD], const u32x4_t (&qB)[kSteps], Request request) {
  if constexpr (AHEAD > 1) unroll_n<AHEAD>([&](auto i) __attribute__((always_inline)) { request(i, frag[decltype(i)::value % AHEAD]); });
  unroll_n<16>([&](auto i) __attribute__((always_inline)) {
    constexpr int f = decltype(i)::value;
    if constexpr (AHEAD == 1) request(i, frag[0]);
    S[f & 1] = mfma32(frag[f % AHEAD], qB[f >> 1], f < 2 ? kZero16 : S[f & 1]);
    if constexpr (AHEAD > 1) {
      request(std::integral_constant<int, f + AHEAD>{}, frag[(f + AHEAD) % AHEAD]);
      __builtin_amdgcn_sched_barrier(0);
    }
  });
}
template <int AHEAD, class Request>
__device__ __forceinline__ void tile_product(f32x16_t (&O)[kDimTiles], u32x4_t (&frag)[AHEAD], const u32x4_t (&pB)[2][2], Request request) {
  unroll_n<16>([&](auto i) __attribute__((always_inline)) {
    constexpr int g = decltype(i)::value, f = 16 + g;
    if constexpr (AHEAD == 1) request(std::integral_constant<int, f>{}, frag[0]);
    O[g & 3] = mfma32(frag[f % AHEAD], pB[g >> 3][(g >> 2) & 1], O[g & 3]);
    if constexpr (AHEAD > 1) {
      if constexpr (f + AHEAD < 32) request(std::integral_constant<int, f + AHEAD>{}, frag[(f + AHEAD) % AHEAD]);
      __builtin_amdgcn_sched_barrier(0);
    }
  });
}

// EXT compiles in the rarely used options (temperature factor, custom mask / no mask); the
// plain causal instantiation keeps its scale in a scalar register and its mask test to one compare.
// HEADS4: the short-chunk tile (chunks of at most 64 tokens: a verify step, a short prompt).  A workgroup owns 32
// query positions of FOUR query heads of a kv head, one head per wave, instead of 128 positions of one head:
// such chunks then fill their tiles, and the four waves still share every K/V tile.
template <bool UNIFORM, bool CAP, bool EXT, bool HEADS4 = false>
__global__ __launch_bounds__(256, 2) void rpa_prefill_async_kernel(const PrefillArgs a_in, int tiles, int nseq, bool by_level) {
  PrefillArgs a = a_in;  // static-shape mode: the sequences to process come from the device
  if (a.dist) {
    a.seq_begin = (a.sm.mask_mode == 1) ? 0 : scalar_load_i32(a.dist);
    a.seq_end = min(a.seq_end, scalar_load_i32(a.dist + 2));
    if (a.seq_begin >= a.seq_end) return;
  }
  // Four separate arrays (not one indexed array): the compiler can then prove that the
  // asynchronous copy into one ring slot does not alias the LDS reads of the other slot and
  // does not drain the vector-memory queue in the middle of a tile.
  __shared__ __attribute__((aligned(1024))) char lds_k0[kTileB];
  __shared__ __attribute__((aligned(1024))) char lds_k1[kTileB];
  __shared__ __attribute__((aligned(1024))) char lds_v0[kTileB];
  __shared__ __attribute__((aligned(1024))) char lds_v1[kTileB];

  constexpr int BM = HEADS4 ? 32 : kBM;  // query positions per workgroup
  Work w = decompose<true>(a, tiles, nseq, by_level, BM, HEADS4 ? 4 : 1);
  if (!w.valid) {
    write_new_tokens(a_in);
    return;
  }
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if constexpr (HEADS4) w.head += wave;  // this wave's head
  const int c = lane & 31, h = lane >> 5;
  const TileSrc src = make_src(a, w);
  const char* kh = head_rows(a, w, a.kv.k_base);
  const char* vh = head_rows(a, w, a.kv.v_base);

  WaveRows wr;
  wr.r_lo = w.q_start + (HEADS4 ? 0 : wave * 32);
  wr.r_hi = min(wr.r_lo + 31, w.q_len - 1);
  wr.active = wr.r_lo < w.q_len;
  wr.row = wr.r_lo + c;
  wr.qpos = w.prefix + wr.row;
  const int W_ = a.sm.window;

  u32x4_t qB[kSteps];
  {
    const int rr = min(wr.row, w.q_len - 1);
    const uint16_t* qp = a.q + ((int64_t)(w.qg0 + rr) * a.Hq + w.head) * a.q_dim;
    ld_query_row<kSteps, kHeadDim>(qB, qp, h, a.q_dim);
    if (EXT && a.sm.q_scale > 0.f) {
#pragma unroll
      for (int ks = 0; ks < kSteps; ++ks) qB[ks] = requantise_q(qB[ks], a.sm.q_scale, false);
    }
  }
  Softmax<CAP> sm;
  sm.scale = a.sm.sm_scale * (a.k_scale ? scalar_load_f32(a.k_scale + w.hk) : 1.0f) *
             ((EXT && a.sm.q_scale > 0.f) ? a.sm.q_scale : 1.0f);
  if constexpr (!CAP) make_scale_positive(sm.scale, qB);
  sm.cap = a.sm.soft_cap;
  sm.inv_cap = (sm.cap != 0.f) ? 1.0f / sm.cap : 0.f;
  {
    const float temp = EXT ? xai_factor(wr.qpos, a.sm.xai_len) : 1.0f;  // per query row
    sm.sc2 = CAP ? 1.0f : sm.scale * kLog2e * temp;
    sm.temp = temp;
    sm.round_mode = a.sm.round_logits;
  }

  f32x16_t O[kDimTiles];
#pragma unroll
  for (int d = 0; d < kDimTiles; ++d)
#pragma unroll
    for (int v = 0; v < 16; ++v) O[d][v] = 0.f;
  float m = kMaxFloor, l = 0.f;

  const int wg_r_hi = min(w.q_start + BM, w.q_len) - 1;
  const bool causal = !EXT || a.sm.mask_mode == 0;
  MaskCtx mc;
  mc.mode = 0;
  if constexpr (EXT) mc = make_mask_ctx(a, w, wr.row);
  int t_hi = causal ? min(w.kv_len, w.prefix + wg_r_hi + 1) : w.kv_len;  // exclusive
  int t_lo = 0;
  if (W_ > 0) t_lo = max(0, w.prefix + w.q_start - W_ + 1) & ~(kBN - 1);
  int split = 0;
  if (a.kv_splits > 1 && !kv_piece(a, t_lo, t_hi, split)) {  // under-filled launch, nothing left for this piece
    write_empty_partial_rows(a, w, wr, h, split);
    return;
  }

  // ---- operand addresses inside a tile (bytes) ----
  // K operand of (m-tile mt, k-step ks): row 32mt + c, chunk (2ks + h) ^ (c & 15)
  const int k_row = c * kRowB;
  const int k_swz = (h ^ (c & 15)) << 4;  // chunk = (2ks) ^ (h ^ (c & 15)), in bytes: (32ks) ^ k_swz
  // V^T operand of (dim tile d, m-tile mt, k-step kk), first / second half of the k-step:
  //   source lane r = lane & 15 of its 16-lane block points at token 32mt + 16kk + 4h + (r >> 2) (+ 8),
  //   dims 32d + 16*(block & 1) + 4*(r & 3); chunk = (4d + 2*(block & 1) + ((r & 3) >> 1)) ^ (4*(r >> 2))
  const int r16 = lane & 15, b16 = lane >> 4;
  const int v_row = (4 * h + (r16 >> 2)) * kRowB;
  const int v_in = ((b16 & 1) << 5) + (((r16 & 3) >> 1) << 4) + ((r16 & 1) << 3);
  const int v_swz = (r16 >> 2) << 6;  // byte offset of the 64-byte window: (64d) ^ v_swz
  // The swizzled offsets are kept in registers for the whole loop (12 of them) instead of being
  // recomputed in front of each of the 48 LDS reads of a tile; slot bases and row steps fold
  // into the instructions' immediate offsets.
  int koff[kSteps], voff[kDimTiles];
#pragma unroll
  for (int ks = 0; ks < kSteps; ++ks) {
    koff[ks] = k_row + ((ks * 32) ^ k_swz);
    asm volatile("" : "+v"(koff[ks]));
  }
#pragma unroll
  for (int d = 0; d < kDimTiles; ++d) {
    voff[d] = v_row + v_in + ((d * 64) ^ v_swz);
    asm volatile("" : "+v"(voff[d]));
  }

  // ---- pipeline: page ids two tiles ahead, the asynchronous copy one tile ahead ----
  RowFeed<16, kCopies> feed;  // UNIFORM: a wave copies 16 rows of a tile
  AsyncPages pg;
  auto feed_row = [&](int n) { return n * kRowsPerCopy + lane / kChunks; };
  auto fetch_pages = [&](int tb) __attribute__((always_inline)) {
    if constexpr (UNIFORM) feed.fetch_page(src, tb, wave);
    else async_fetch_pages(pg, src, tb, wave, lane);
  };
  auto copy_tile = [&](char* to_k, char* to_v, int tb) __attribute__((always_inline)) {
    if constexpr (UNIFORM) {
      typedef __attribute__((address_space(3))) char* at_t;
      const int64_t base = feed.base(src, a.kv);
      feed.template copy<false>((uint32_t)(uintptr_t)(at_t)to_k + wave * (kCopies * 1024), kh + base, src, a.kv, feed_row);
      feed.template copy<true>((uint32_t)(uintptr_t)(at_t)to_v + wave * (kCopies * 1024), vh + base, src, a.kv, feed_row);
    } else {
      async_copy_tile(to_k, to_v, src, a.kv, kh, vh, tb, wave, lane, pg);
    }
  };
  if constexpr (UNIFORM)
    feed.init(a.kv, feed_row, [&](int n) { return (lane % kChunks) ^ (feed_row(n) & 15); },
              [&](int n) { return (lane % kChunks) ^ ((feed_row(n) & 3) << 2); });
  fetch_pages(t_lo);
  copy_tile(lds_k0, lds_v0, t_lo);
  fetch_pages(t_lo + kBN);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the copies have landed in LDS
  __syncthreads();

  // one tile: consume (lds_k, lds_v), fill (nxt_k, nxt_v) with the tile after it
  auto tile_step = [&](const char* lds_k, const char* lds_v, char* nxt_k, char* nxt_v, int tb) {
    uint64_t mask_word = 0;  // a caller's mask turned into bits by the pre-pass: one word per lane and tile
    if constexpr (EXT) {
      if (mc.mode == 1 && mc.bits) mask_word = mc.bits[min(tb >> 6, mc.bit_words - 1)];
    }
    if (tb + kBN < t_hi) {
      // the other slot was last read before the barrier that ended the previous tile
      copy_tile(nxt_k, nxt_v, tb + kBN);
      fetch_pages(tb + 2 * kBN);
    }
    // visible to this wave?  causal: some token <= last row's position; window: some token
    // newer than the first row's horizon
    const bool vis = wr.active && (!causal || tb <= w.prefix + wr.r_hi) &&
                     (W_ <= 0 || tb + kBN - 1 > w.prefix + wr.r_lo - W_);
    if (vis) {
      const bool need_mask = (causal ? (tb + kBN - 1 > w.prefix + wr.r_lo) : (mc.mode == 1 || tb + kBN > w.kv_len)) ||
                             (W_ > 0 && tb <= w.prefix + wr.r_hi - W_);
      auto request = [&](auto tag, u32x4_t& to) __attribute__((always_inline)) {
        constexpr int f = decltype(tag)::value;
        if constexpr (f < 16) {
          to = lds_ld16(lds_k + koff[f >> 1] + (f & 1) * (32 * kRowB));
        } else {
          const char* vt = lds_v + voff[f & 3] + (((f >> 3) & 1) * 32 + ((f >> 2) & 1) * 16) * kRowB;
          const u32x2_t lo = lds_tr16(vt), hi = lds_tr16(vt + 8 * kRowB);
          to = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
        }
      };
      f32x16_t S[2];
      u32x4_t frag[EXT ? 2 : UNIFORM ? 6 : 4];
      tile_scores(S, frag, qB, request);
      u32x4_t pB[2][2];
      softmax_tile<CAP, EXT>(S, O, m, l, sm, need_mask, tb, h, wr.qpos, W_, pB, mc, mask_word);
      tile_product(O, frag, pB, request);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // the next tile has landed
    __syncthreads();
  };
  for (int tb = t_lo; tb < t_hi; tb += 2 * kBN) {
    tile_step(lds_k0, lds_v0, lds_k1, lds_v1, tb);
    if (tb + kBN >= t_hi) break;
    tile_step(lds_k1, lds_v1, lds_k0, lds_v0, tb + kBN);
  }
  if (a.kv_splits > 1) write_partial_rows(a, w, wr, O, l, h, m * sm.sc2, split);
  else write_rows(a, w, wr, O, l, h, m * sm.sc2);
}

}  // namespace

// ==================================================================== 256-wide heads
// A workgroup owns 128 query positions of one query head with EIGHT waves of 16 positions (16x16x32 matrix
// instructions), two waves per SIMD.  A wave holds Q^T of its positions (32 registers), O^T (64), the scores of a 64-token
// tile (16) and the probabilities of the one before.  With four waves of 32 positions and 512 registers, what was here
// before, a lone wave per SIMD had its operand reads and its exponentials exposed, and the compiler moved operands through
// the accumulation registers and drained the loads in flight to make room.  The price is LDS: every wave reads the whole
// K and V tile, 512 KiB per tile and CU, 2300 clocks (3.7 per ds_read_b128, 2.6 per transposing read) against 2048 of the
// matrix pipe.  Counters (e4m3, soft cap, window): LDS 27 %, vector pipe 26 %, matrix pipe 17 % of the launch's clocks, for
// 64 % of which the CUs hold their waves (704 workgroups on 256 CUs pack badly): no pipe is full, the waves of a CU go
// through its phases together.
// (Eight waves as pairs that share 32 positions, one set of scores each, and exchange their probabilities through LDS --
// half the reads -- spilled 50 registers at 256: 423 us.)
// Measured: 6 chunks of 300 .. 1500 tokens x 16 heads, e4m3, soft cap, window 1024 (89 GFLOP) 424 -> 193 us; 3 bf16 prompts of
// 1490 .. 2883 tokens x 16 heads on 16-token pages 198 -> 137 us with the cache write.
namespace {

constexpr int kWRowB = 512;                // a K or V row in LDS
constexpr int kWTileB = kBN * kWRowB;      // 32 KiB
typedef __attribute__((address_space(3))) char* lds_ptr_t;  // the ring is addressed by offset: a tile's halves are an xor apart

__device__ __forceinline__ u32x4_t ring_ld16(uint32_t at) {
  return *reinterpret_cast<__attribute__((address_space(3))) const u32x4_t*>((lds_ptr_t)(uintptr_t)at);
}
__device__ __forceinline__ void ring_st16(uint32_t at, u32x4_t v) {
  *reinterpret_cast<__attribute__((address_space(3))) u32x4_t*>((lds_ptr_t)(uintptr_t)at) = v;
}
__device__ __forceinline__ u32x2_t ring_tr16(uint32_t at) {
  typedef __attribute__((address_space(3))) s16x4_t* ptr_t;
  return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr_t)(uintptr_t)at));
}
__device__ __forceinline__ const void* ring_ptr(uint32_t at) { return (const void*)(lds_ptr_t)(uintptr_t)at; }

// bf16 rows: every wave copies 4 x 64 chunks of 16 bytes of K and of V (two rows per copy instruction); chunk j of row t
// sits at chunk position j ^ swizzle(t), K: t & 15, V: 4 (t & 3) + 2 ((t >> 2) & 1) -- 32 lanes of a transposing read
// meet rows t .. t + 7 in the same 32 bytes, and every bank once.
// e4m3 rows: their bytes arrive in LDS as they are, two tiles ahead, in an area of the wave's own (2 x 1 KiB of K, of V):
// a lane copies the 16 bytes that it later widens, so nothing but the wave's own wait stands between the two and no
// register holds them on the way.  Piece p of a row (16 bytes) widens to chunks 2p and 2p + 1.
__device__ __forceinline__ int wide_v_swizzle(int t) { return ((t & 3) << 2) | ((t >> 1) & 2); }

template <bool UNIFORM, bool FP8>
struct WideFeed {
  static constexpr int N = FP8 ? 2 : 4;  // copy instructions per wave, for K and for V
  RowFeed<8, N> rows;                    // UNIFORM: a wave copies 8 rows of a tile
  int32_t id[N];                         // else: pages of this lane's rows in the tile copied next

  __device__ __forceinline__ static int row(int n, int wave, int lane) {
    return FP8 ? wave * 8 + n * 4 + (lane >> 4) : wave * 8 + n * 2 + (lane >> 5);
  }
  __device__ __forceinline__ static int own_row(int n, int lane) { return FP8 ? n * 4 + (lane >> 4) : n * 2 + (lane >> 5); }
  __device__ __forceinline__ void init(const KvAddr& kv, int wave, int lane) {
    if constexpr (UNIFORM)
      rows.init(kv, [&](int n) { return own_row(n, lane); },
                [&](int n) { return FP8 ? (lane & 15) : (lane & 31) ^ (row(n, wave, lane) & 15); },
                [&](int n) { return FP8 ? (lane & 15) : (lane & 31) ^ wide_v_swizzle(row(n, wave, lane)); });
  }
  __device__ __forceinline__ void fetch_pages(const TileSrc& s, int tb, int wave, int lane) {
    if constexpr (UNIFORM) {
      rows.fetch_page(s, tb, wave);
    } else {
      tb = min(tb, s.last_tok & ~(kBN - 1));
#pragma unroll
      for (int n = 0; n < N; ++n) id[n] = s.pages[page_slot(s, min(tb + row(n, wave, lane), s.last_tok))];
    }
  }
  // K (or V) rows to `at` (FP8: the bytes to the staging area at `at`)
  __device__ __forceinline__ void copy(bool is_v, uint32_t at, const TileSrc& s, const KvAddr& kv, const char* base, int tb, int wave,
                                       int lane) {
    if constexpr (UNIFORM) {
      const char* b = base + rows.base(s, kv);
      auto own = [&](int n) { return own_row(n, lane); };
      if (is_v) rows.template copy<true>(at + wave * (N * 1024), b, s, kv, own);
      else rows.template copy<false>(at + wave * (N * 1024), b, s, kv, own);
      return;
    }
    tb = min(tb, s.last_tok & ~(kBN - 1));  // past the end: re-copy the last tile
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int t = row(n, wave, lane);
      const int64_t ro = row_offset<false>(s, kv, tb, tb + t, id[n]);
      const int j = FP8 ? (lane & 15) : (lane & 31) ^ (is_v ? wide_v_swizzle(t) : t & 15);
      async_copy16(base + ro + j * 16, ring_ptr(at + (wave * N + n) * 1024));
    }
  }
  // FP8: the staged bytes of this wave's rows -> bf16 rows of a tile (16 lanes of a row write chunks two apart: all banks)
  __device__ __forceinline__ static void widen(uint32_t stage, uint32_t at, bool is_v, int wave, int lane) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int t = row(n, wave, lane), j = 2 * (lane & 15), swz = is_v ? wide_v_swizzle(t) : t & 15;
      const u32x4_t x = ring_ld16(stage + (wave * N + n) * 1024 + lane * 16);
      const u32x2_t a = fp8x4_to_bf16x4(x[0]), b = fp8x4_to_bf16x4(x[1]), c = fp8x4_to_bf16x4(x[2]), d = fp8x4_to_bf16x4(x[3]);
      ring_st16(at + t * kWRowB + ((j ^ swz) << 4), u32x4_t{a[0], a[1], b[0], b[1]});
      ring_st16(at + t * kWRowB + (((j + 1) ^ swz) << 4), u32x4_t{c[0], c[1], d[0], d[1]});
    }
  }
};

template <bool UNIFORM, bool CAP, bool EXT, bool FP8>
__global__ __launch_bounds__(512, 2) void rpa_prefill_async_kernel_wide(const PrefillArgs a_in, int tiles, int nseq, bool by_level) {
  PrefillArgs a = a_in;  // static-shape mode: the sequences to process come from the device
  if (a.dist) {
    a.seq_begin = (a.sm.mask_mode == 1) ? 0 : scalar_load_i32(a.dist);
    a.seq_end = min(a.seq_end, scalar_load_i32(a.dist + 2));
    if (a.seq_begin >= a.seq_end) return;
  }
  __shared__ __attribute__((aligned(65536))) char ring[4 * kWTileB];  // K, K, V, V
  __shared__ __attribute__((aligned(1024))) char stage[FP8 ? kWTileB : 16];  // K bytes, V bytes

  const Work w = decompose(a, tiles, nseq, by_level, kBM, 1);
  if (!w.valid) {
    write_new_tokens(a_in);
    return;
  }
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const TileSrc src = make_src(a, w);
  const char* kh = head_rows(a, w, a.kv.k_base);
  const char* vh = head_rows(a, w, a.kv.v_base);

  // this wave's positions: [r_lo, r_hi] of the chunk, lane column c = position r_lo + c
  const int r_lo = w.q_start + wave * 16, r_hi = min(r_lo + 15, w.q_len - 1);
  const bool active = r_lo < w.q_len;
  const int row = r_lo + c, qpos = w.prefix + row;
  const int W_ = a.sm.window;

  const int wg_r_hi = min(w.q_start + kBM, w.q_len) - 1;
  const bool causal = !EXT || a.sm.mask_mode == 0;
  MaskCtx mc;
  mc.mode = 0;
  if constexpr (EXT) mc = make_mask_ctx(a, w, row);
  int t_hi = causal ? min(w.kv_len, w.prefix + wg_r_hi + 1) : w.kv_len;  // exclusive
  int t_lo = 0;
  if (W_ > 0) t_lo = max(0, w.prefix + w.q_start - W_ + 1) & ~(kBN - 1);
  int split = 0;
  if (a.kv_splits > 1 && !kv_piece(a, t_lo, t_hi, split)) t_hi = t_lo;  // under-filled launch, nothing left for this piece

  // ---- Q^T operands: column c = position, k-step ks covers dims 32 ks + 8 g ..
  u32x4_t qB[8];
  {
    const uint16_t* qp = a.q + ((int64_t)(w.qg0 + min(row, w.q_len - 1)) * a.Hq + w.head) * a.q_dim;
    ld_query_row<8, 256>(qB, qp, g, a.q_dim);
  }

  // ---- the first tiles are asked for with the queries, in one round trip (their order: see below); e4m3: the second tile's K bytes
  // wait where its V rows will be.  As three trips, queries, first tile, second tile, the chunks above took 189.0 us instead of 188.0, 3
  // bf16 prompts on 16-token pages 148.5 instead of 146.9; with the queries behind the tiles bf16 lost 1 %.
  const uint32_t ring_at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)ring);
  const uint32_t stage_k = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)stage), stage_v = stage_k + kWTileB / 2;
  WideFeed<UNIFORM, FP8> fk, fv;  // the page ids of the K and V copied next
  if (t_lo < t_hi) {
    fk.init(a.kv, wave, lane);
    fv.init(a.kv, wave, lane);
    fk.fetch_pages(src, t_lo, wave, lane);
    fv.fetch_pages(src, t_lo + kBN, wave, lane);
    if constexpr (FP8) {
      fk.copy(false, stage_k, src, a.kv, kh, t_lo, wave, lane);
      fk.copy(true, stage_v, src, a.kv, vh, t_lo, wave, lane);
      fv.copy(false, ring_at + 3 * kWTileB, src, a.kv, kh, t_lo + kBN, wave, lane);
    } else {
      fk.copy(false, ring_at, src, a.kv, kh, t_lo, wave, lane);
      fk.copy(true, ring_at + 2 * kWTileB, src, a.kv, vh, t_lo, wave, lane);
      fv.copy(false, ring_at + kWTileB, src, a.kv, kh, t_lo + kBN, wave, lane);
    }
    fk.fetch_pages(src, t_lo + 2 * kBN, wave, lane);
  }

  if (EXT && a.sm.q_scale > 0.f) {
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qB[ks] = requantise_q(qB[ks], a.sm.q_scale, FP8);
  }
  float scale = a.sm.sm_scale * (a.k_scale ? scalar_load_f32(a.k_scale + w.hk) : 1.0f) * ((EXT && a.sm.q_scale > 0.f) ? a.sm.q_scale : 1.0f);
  if constexpr (!CAP) make_scale_positive(scale, qB);
  const float temp = EXT ? xai_factor(qpos, a.sm.xai_len) : 1.0f;  // per position
  const float sc2 = CAP ? 1.0f : scale * kLog2e * temp;            // score -> log2 units (soft-capped scores are there already)

  f32x4_t O[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) O[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = kMaxFloor, l = 0.f;

  // ---- operand addresses: K row 16 b + c, chunk (4 ks + g) ^ c; V^T of dims 16 j .., token 4 g + (c >> 2) (+ 16 for the
  // second half of the k-step): chunk 2 j + ((c & 3) >> 1) before the swizzle, 8 bytes (c & 1) of it
  uint32_t koff[4], voff[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) koff[i] = ring_at + c * kWRowB + (((4 * i + g) ^ c) << 4);  // steps 4 .. 7: 256 bytes on
#pragma unroll
  for (int i = 0; i < 8; ++i)  // dims 128 ..: 256 bytes on
    voff[i] = ring_at + 2 * kWTileB + (4 * g + (c >> 2)) * kWRowB + (((2 * i + ((c & 3) >> 1)) ^ ((c >> 2) << 2) ^ ((g & 1) << 1)) << 4) + ((c & 1) << 3);

  auto scores = [&](f32x4_t (&S)[4]) __attribute__((always_inline)) {  // tokens 16 b + 4 g + r
#pragma unroll
    for (int b = 0; b < 4; ++b) S[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
#pragma unroll
      for (int b = 0; b < 4; ++b) S[b] = mfma16(ring_ld16(koff[ks & 3] + (ks >> 2) * 256 + b * (16 * kWRowB)), qB[ks], S[b]);
#pragma unroll
    for (int i = 0; i < 4; ++i) koff[i] ^= kWTileB;
  };
  auto cap_scores = [&](f32x4_t (&S)[4]) __attribute__((always_inline)) {
    if constexpr (CAP) {
      const float cap = a.sm.soft_cap;
      if (cap != 0.f && !a.sm.round_logits) {
        // cap tanh(s scale / cap) temp log2e = k2 - 2 k2 / (2^(s k1) + 1)
        const float k1 = scale / cap * (2.0f * kLog2e), k2 = cap * temp * kLog2e;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            S[b][r] = __builtin_fmaf(__builtin_amdgcn_rcpf(fast_exp2(S[b][r] * k1) + 1.0f), -2.0f * k2, k2);
      } else {
        const float inv_cap = cap != 0.f ? 1.0f / cap : 0.f;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float x = S[b][r] * scale;
            if (cap != 0.f) x = soft_cap_f(x, cap, inv_cap);
            x = x * temp;
            if (a.sm.round_logits) x = round_logit(x, a.sm.round_logits);
            S[b][r] = x * kLog2e;
          }
      }
    }
  };
  auto mask_scores = [&](f32x4_t (&S)[4], int tb) __attribute__((always_inline)) {
    if ((causal ? (tb + kBN - 1 > w.prefix + r_lo) : (mc.mode == 1 || tb + kBN > w.kv_len)) ||
        (W_ > 0 && tb <= w.prefix + r_hi - W_)) {
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int tok = tb + 16 * b + 4 * g + r;
          bool masked;
          if (!EXT || mc.mode == 0) masked = tok > qpos;
          else masked = (tok >= mc.kv_len) || (mc.mode == 1 && mc.row[tok] < 1);
          masked = masked || (W_ > 0 && tok <= qpos - W_);
          S[b][r] = masked ? kMaskRaw : S[b][r];
        }
    }
  };
  // probabilities as bf16 pairs, the B operands of the second product; the row sum is taken over the rounded pairs
  u32x4_t pB[2];
  auto probabilities = [&](const f32x4_t (&S)[4], u32x4_t (&p)[2]) __attribute__((always_inline)) {
    const float neg_m = -m * sc2;
    const bf16x2_t ones = {(__bf16)1.0f, (__bf16)1.0f};
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        const uint32_t x = pack_bf16x2(fast_exp2(__builtin_fmaf(S[b][r], sc2, neg_m)), fast_exp2(__builtin_fmaf(S[b][r + 1], sc2, neg_m)));
        l = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, x), ones, l, false);
        p[b >> 1][(b & 1) * 2 + (r >> 1)] = x;
      }
  };
  // The running max goes stale by up to 2^kMaxSlack before what was taken against it follows (see softmax_tile).  The
  // probabilities whose half of the second product is still to come are bf16 and stay what they are (multiplied here they
  // would be rounded again, which l would not): O follows behind that product, when the caller multiplies it by the
  // factor returned.
  auto raise_max = [&](const f32x4_t (&S)[4]) __attribute__((always_inline)) -> float {
    float mx = fmaxf(S[0][0], S[0][1]);
#pragma unroll
    for (int i = 2; i < 16; i += 2) mx = __builtin_fmaxf(__builtin_fmaxf(mx, S[i >> 2][i & 3]), S[i >> 2][(i & 3) + 1]);
    mx = swap_max(swap16_max(mx));
    float alpha = 1.0f;
    if (__builtin_amdgcn_ballot_w64((mx - m) * sc2 > kMaxSlack) != 0) {
      const float m_new = fmaxf(m, mx);
      alpha = fast_exp2((m - m_new) * sc2);
      m = m_new;
      l *= alpha;
    }
    return alpha;
  };
  auto second_product = [&](int kk) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const uint32_t vt = voff[j & 7] + (j >> 3) * 256 + kk * (32 * kWRowB);
      const u32x2_t lo = ring_tr16(vt);
      const u32x2_t hi = ring_tr16(vt + 16 * kWRowB);
      O[j] = mfma16(u32x4_t{lo[0], lo[1], hi[0], hi[1]}, pB[kk], O[j]);
    }
  };

  // ---- a step's 64 operand fragments in the order of their use -- K of the scores (f < 32), V^T of the two halves of the
  // second product -- kAhead of them requested ahead of the matrix instruction that takes them, across the softmax in between.
  // (Left to itself the compiler asks for two at a time and waits: 203.5 -> 193 us on the chunks above, 2 chunks of 1024 on 2048,
  // bf16, 125.7 -> 113.1; 4, 8 or 10 ahead are the same.)
  constexpr int kAhead = 6;
  u32x4_t frag[kAhead];
  auto request = [&](auto tag) __attribute__((always_inline)) {
    constexpr int f = decltype(tag)::value;
    if constexpr (f < 32) {
      frag[f % kAhead] = ring_ld16(koff[(f >> 2) & 3] + (f >> 4) * 256 + (f & 3) * (16 * kWRowB));
    } else if constexpr (f < 64) {
      const uint32_t vt = voff[f & 7] + ((f & 15) >> 3) * 256 + ((f - 32) >> 4) * (32 * kWRowB);
      const u32x2_t lo = ring_tr16(vt), hi = ring_tr16(vt + 16 * kWRowB);
      frag[f % kAhead] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
    }
  };
  auto scores_of = [&](f32x4_t (&S)[4]) __attribute__((always_inline)) {
    unroll_n<kAhead>([&](auto i) __attribute__((always_inline)) { request(i); });
    unroll_n<32>([&](auto i) __attribute__((always_inline)) {
      constexpr int f = decltype(i)::value;
      S[f & 3] = mfma16(frag[f % kAhead], qB[f >> 2], f < 4 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : S[f & 3]);
      request(std::integral_constant<int, f + kAhead>{});
      __builtin_amdgcn_sched_barrier(0);
    });
#pragma unroll
    for (int i = 0; i < 4; ++i) koff[i] ^= kWTileB;
  };
  auto product_half = [&](auto half) __attribute__((always_inline)) {
    constexpr int kk = decltype(half)::value;
    unroll_n<16>([&](auto i) __attribute__((always_inline)) {
      constexpr int j = decltype(i)::value, f = 32 + 16 * kk + j;
      O[j] = mfma16(frag[f % kAhead], pB[kk], O[j]);
      request(std::integral_constant<int, f + kAhead>{});
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  // ---- K runs a tile ahead of V.  Step i: K of tile i + 2 and V of tile i + 1 are requested; scores of tile i + 1, whose
  // soft cap and exponentials run beside the two halves of the second product of tile i
  if (t_lo < t_hi) {
    const int n = __builtin_amdgcn_readfirstlane((t_hi - t_lo + kBN - 1) / kBN);
    uint32_t k_fill = ring_at, v_fill = ring_at + 3 * kWTileB;
    wait_all_loads();
    if constexpr (FP8) {
      fk.widen(stage_k, ring_at, false, wave, lane);
      fk.widen(stage_v, ring_at + 2 * kWTileB, true, wave, lane);
      fk.widen(ring_at + 3 * kWTileB, ring_at + kWTileB, false, wave, lane);
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the bytes have been read
      fv.copy(true, stage_v, src, a.kv, vh, t_lo + kBN, wave, lane);
      fk.copy(false, stage_k, src, a.kv, kh, t_lo + 2 * kBN, wave, lane);
      fv = fk;
      fk.fetch_pages(src, t_lo + 3 * kBN, wave, lane);
    }
    __syncthreads();
    auto next = [&](int tb) __attribute__((always_inline)) {
      if constexpr (FP8) {
        wait_all_loads();  // this wave's bytes: K of tile i + 2, V of tile i + 1
        fk.widen(stage_k, k_fill, false, wave, lane);
        fk.widen(stage_v, v_fill, true, wave, lane);
        __builtin_amdgcn_s_waitcnt(0xC07F);
        fk.copy(false, stage_k, src, a.kv, kh, tb + 3 * kBN, wave, lane);
        fv.copy(true, stage_v, src, a.kv, vh, tb + 2 * kBN, wave, lane);
        fv = fk;
        fk.fetch_pages(src, tb + 4 * kBN, wave, lane);
      } else {
        fk.copy(false, k_fill, src, a.kv, kh, tb + 2 * kBN, wave, lane);
        fv.copy(true, v_fill, src, a.kv, vh, tb + kBN, wave, lane);
        fv = fk;
        fk.fetch_pages(src, tb + 3 * kBN, wave, lane);
      }
      k_fill ^= kWTileB;
      v_fill ^= kWTileB;
    };
    auto meet = [&]() __attribute__((always_inline)) {
      if constexpr (!FP8) wait_all_loads();  // this wave's copies have landed
      __syncthreads();
    };
    if (__builtin_amdgcn_readfirstlane(!active)) {  // positions past the chunk's end: this wave only copies
      for (int i = 0; i + 1 < n; ++i) {
        if (i == 0) __syncthreads();
        next(t_lo + i * kBN);
        meet();
      }
    } else {
      {
        f32x4_t S[4];
        scores(S);
        cap_scores(S);
        mask_scores(S, t_lo);
        raise_max(S);  // (O is zero)
        probabilities(S, pB);
      }
      // (tiles that none of a wave's positions sees are not skipped: the other waves of the workgroup are at work on them)
      for (int i = 0; i + 1 < n; ++i) {
        const int tb = t_lo + i * kBN;
        // (K of tile 0 is free once every wave has taken its scores of it)
        if (i == 0) __syncthreads();
        next(tb);
        f32x4_t S[4];
        scores_of(S);
        cap_scores(S);
        product_half(std::integral_constant<int, 0>{});
        mask_scores(S, tb + kBN);
        const float alpha = raise_max(S);
        u32x4_t p_next[2];
        probabilities(S, p_next);
        product_half(std::integral_constant<int, 1>{});
        pB[0] = p_next[0];
        pB[1] = p_next[1];
#pragma unroll
        for (int k = 0; k < 8; ++k) voff[k] ^= kWTileB;
        // (here and not right behind the product: 3 bf16 prompts 153.7 -> 151.4 us, 64-token pages 375.6 -> 377.6)
        if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
          for (int j = 0; j < 16; ++j) O[j] *= alpha;
        }
        meet();
      }
      second_product(0);
      second_product(1);
    }
    if constexpr (FP8) wait_all_loads();  // (bytes requested past the end)
  }

  // ---- lane (c, g) holds position r_lo + c, dims 16 j + 4 g + r
  l = swap_sum(swap16_sum(l));
  if (!active) return;
  const bool real = row < w.q_len;
  const int64_t out_row = (int64_t)(w.qg0 + row) * a.Hq + w.head;
  if (a.kv_splits > 1) {
    if (!real) return;
    const int64_t slot = out_row * a.kv_splits + split;
    float* op = a.ws_o + slot * 256 + 4 * g;
#pragma unroll
    for (int j = 0; j < 16; ++j) *reinterpret_cast<f32x4_t*>(op + 16 * j) = O[j];
    if (g == 0) {
      a.ws_ml[slot * 2] = fmaxf(m * sc2, kNoReference);
      a.ws_ml[slot * 2 + 1] = l;
    }
    return;
  }
  const float vs = a.v_scale ? scalar_load_f32(a.v_scale + w.hk) : 1.0f;
  const float inv = a.sm.sink ? vs * sink_inverse(m * sc2, l, sink_logit(a.sm.sink, a.sm.round_logits, w.head)) : vs / l;
  uint16_t* op = a.out + out_row * a.q_dim + 8 * g;
#pragma unroll
  for (int j = 0; j < 16; j += 2) {
    const u32x4_t o = row_of_16(u32x2_t{pack_bf16x2(O[j][0] * inv, O[j][1] * inv), pack_bf16x2(O[j][2] * inv, O[j][3] * inv)},
                                u32x2_t{pack_bf16x2(O[j + 1][0] * inv, O[j + 1][1] * inv), pack_bf16x2(O[j + 1][2] * inv, O[j + 1][3] * inv)});
    if (real && 16 * j + 8 * g < a.q_dim) st16(op + 16 * j, o);
  }
}

}  // namespace

namespace {

// ==================================================================== staged path (fp8 cache)
constexpr int kKPitch = 272;  // bytes per K row in LDS (256 + 16 pad: conflict-free b128 reads)
constexpr int kVPitch = 144;  // bytes per V^T row in LDS (128 + 16 pad)

template <bool UNIFORM>
struct PageIds {
  int32_t id[UNIFORM ? 1 : 8];
};

template <bool FP8>
struct Stage {
  u32x4_t r[FP8 ? 4 : 8];
};

template <bool UNIFORM>
__device__ __forceinline__ void fetch_page_ids(PageIds<UNIFORM>& pg, const TileSrc& s, int tb, int tid) {
  tb = min(tb, s.last_tok & ~(kBN - 1));
  if constexpr (UNIFORM) {
    pg.id[0] = scalar_load_i32(s.pages + __builtin_amdgcn_readfirstlane(page_slot(s, tb)));
  } else {
    if (tid < 128) {
      pg.id[0] = s.pages[page_slot(s, min(tb + (tid >> 1), s.last_tok))];
    } else {
      const int tg = (tid - 128) & 7;
#pragma unroll
      for (int i = 0; i < 8; ++i) pg.id[i] = s.pages[page_slot(s, min(tb + vt_token(tg, i), s.last_tok))];
    }
  }
}

// Threads 0..127 stage K (one half row each), threads 128..255 stage V (8 tokens x 8 dims each).
template <bool FP8, bool UNIFORM>
__device__ __forceinline__ void tile_gload(Stage<FP8>& st, const TileSrc& s, const KvAddr& kv, const char* kh,
                                           const char* vh, int tb, int tid, const PageIds<UNIFORM>& pg) {
  tb = min(tb, s.last_tok & ~(kBN - 1));  // past the end: re-read the last tile
  if (tid < 128) {
    const int tl = tid >> 1, half = tid & 1;
    const char* p = kh + row_offset<UNIFORM>(s, kv, tb, tb + tl, pg.id[0]) + half * (FP8 ? 64 : 128);
#pragma unroll
    for (int i = 0; i < (FP8 ? 4 : 8); ++i) st.r[i] = ld16(p + i * 16);
  } else {
    const int u = tid - 128;
    const int tg = u & 7, dc = u >> 3;
    if constexpr (FP8) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const u32x2_t x =
            ld8(vh + row_offset<UNIFORM>(s, kv, tb, tb + vt_token(tg, i), pg.id[UNIFORM ? 0 : i]) + dc * 8);
        st.r[i >> 1][(i & 1) * 2 + 0] = x[0];
        st.r[i >> 1][(i & 1) * 2 + 1] = x[1];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        st.r[i] = ld16(vh + row_offset<UNIFORM>(s, kv, tb, tb + vt_token(tg, i), pg.id[UNIFORM ? 0 : i]) + dc * 16);
    }
  }
}

template <bool FP8>
__device__ __forceinline__ void tile_lstore(const Stage<FP8>& st, char* lds_k, char* lds_v, int tid) {
  if (tid < 128) {
    const int tl = tid >> 1, half = tid & 1;
    char* p = lds_k + tl * kKPitch + half * 128;
    if constexpr (FP8) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const u32x2_t a = fp8x4_to_bf16x4(st.r[i][0]);
        const u32x2_t b = fp8x4_to_bf16x4(st.r[i][1]);
        const u32x2_t c = fp8x4_to_bf16x4(st.r[i][2]);
        const u32x2_t d = fp8x4_to_bf16x4(st.r[i][3]);
        lds_st16(p + i * 32, u32x4_t{a[0], a[1], b[0], b[1]});
        lds_st16(p + i * 32 + 16, u32x4_t{c[0], c[1], d[0], d[1]});
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) lds_st16(p + i * 16, st.r[i]);
    }
  } else {
    const int u = tid - 128;
    const int tg = u & 7, dc = u >> 3;
    char* p = lds_v + (dc * 8) * kVPitch + tg * 16;
    if constexpr (FP8) {
      float f[8][8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t w0 = st.r[i >> 1][(i & 1) * 2 + 0];
        const uint32_t w1 = st.r[i >> 1][(i & 1) * 2 + 1];
        const f32x2_t a0 = __builtin_amdgcn_cvt_pk_f32_fp8(w0, false);
        const f32x2_t a1 = __builtin_amdgcn_cvt_pk_f32_fp8(w0, true);
        const f32x2_t a2 = __builtin_amdgcn_cvt_pk_f32_fp8(w1, false);
        const f32x2_t a3 = __builtin_amdgcn_cvt_pk_f32_fp8(w1, true);
        f[i][0] = a0[0]; f[i][1] = a0[1]; f[i][2] = a1[0]; f[i][3] = a1[1];
        f[i][4] = a2[0]; f[i][5] = a2[1]; f[i][6] = a3[0]; f[i][7] = a3[1];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
        lds_st16(p + j * kVPitch, u32x4_t{pack_bf16x2(f[0][j], f[1][j]), pack_bf16x2(f[2][j], f[3][j]),
                                          pack_bf16x2(f[4][j], f[5][j]), pack_bf16x2(f[6][j], f[7][j])});
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
        const int jj = j >> 1;
        lds_st16(p + j * kVPitch,
                 u32x4_t{__builtin_amdgcn_perm(st.r[1][jj], st.r[0][jj], sel),
                         __builtin_amdgcn_perm(st.r[3][jj], st.r[2][jj], sel),
                         __builtin_amdgcn_perm(st.r[5][jj], st.r[4][jj], sel),
                         __builtin_amdgcn_perm(st.r[7][jj], st.r[6][jj], sel)});
      }
    }
  }
}

template <bool FP8, bool UNIFORM, bool CAP, bool EXT, bool HEADS4 = false>
__global__ __launch_bounds__(256, 2) void rpa_prefill_staged_kernel(const PrefillArgs a_in, int tiles, int nseq, bool by_level) {
  PrefillArgs a = a_in;  // static-shape mode: the sequences to process come from the device
  if (a.dist) {
    a.seq_begin = (a.sm.mask_mode == 1) ? 0 : scalar_load_i32(a.dist);
    a.seq_end = min(a.seq_end, scalar_load_i32(a.dist + 2));
    if (a.seq_begin >= a.seq_end) return;
  }
  __shared__ __attribute__((aligned(16))) char lds_k_buf[2][kBN * kKPitch];
  __shared__ __attribute__((aligned(16))) char lds_v_buf[2][128 * kVPitch];

  constexpr int BM = HEADS4 ? 32 : kBM;  // the short-chunk tile: 32 positions x 4 heads, one head per wave
  Work w = decompose<true>(a, tiles, nseq, by_level, BM, HEADS4 ? 4 : 1);
  if (!w.valid) {
    write_new_tokens(a_in);
    return;
  }
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  if constexpr (HEADS4) w.head += wave;
  const int c = lane & 31, h = lane >> 5;
  const TileSrc src = make_src(a, w);
  const char* kh = head_rows(a, w, a.kv.k_base);
  const char* vh = head_rows(a, w, a.kv.v_base);

  WaveRows wr;
  wr.r_lo = w.q_start + (HEADS4 ? 0 : wave * 32);
  wr.r_hi = min(wr.r_lo + 31, w.q_len - 1);
  wr.active = wr.r_lo < w.q_len;
  wr.row = wr.r_lo + c;
  wr.qpos = w.prefix + wr.row;
  const int W_ = a.sm.window;

  u32x4_t qB[8];
  {
    const int rr = min(wr.row, w.q_len - 1);
    const uint16_t* qp = a.q + ((int64_t)(w.qg0 + rr) * a.Hq + w.head) * a.q_dim;
    ld_query_row<8, 128>(qB, qp, h, a.q_dim);
    if (EXT && a.sm.q_scale > 0.f) {
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) qB[ks] = requantise_q(qB[ks], a.sm.q_scale, FP8);
    }
  }
  Softmax<CAP> sm;
  sm.scale = a.sm.sm_scale * (a.k_scale ? scalar_load_f32(a.k_scale + w.hk) : 1.0f) *
             ((EXT && a.sm.q_scale > 0.f) ? a.sm.q_scale : 1.0f);
  if constexpr (!CAP) make_scale_positive(sm.scale, qB);
  sm.cap = a.sm.soft_cap;
  sm.inv_cap = (sm.cap != 0.f) ? 1.0f / sm.cap : 0.f;
  {
    const float temp = EXT ? xai_factor(wr.qpos, a.sm.xai_len) : 1.0f;  // per query row
    sm.sc2 = CAP ? 1.0f : sm.scale * kLog2e * temp;
    sm.temp = temp;
    sm.round_mode = a.sm.round_logits;
  }

  f32x16_t O[4];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int v = 0; v < 16; ++v) O[d][v] = 0.f;
  float m = kMaxFloor, l = 0.f;

  const int wg_r_hi = min(w.q_start + BM, w.q_len) - 1;
  const bool causal = !EXT || a.sm.mask_mode == 0;
  MaskCtx mc;
  mc.mode = 0;
  if constexpr (EXT) mc = make_mask_ctx(a, w, wr.row);
  int t_hi = causal ? min(w.kv_len, w.prefix + wg_r_hi + 1) : w.kv_len;  // exclusive
  int t_lo = 0;
  if (W_ > 0) t_lo = max(0, w.prefix + w.q_start - W_ + 1) & ~(kBN - 1);
  int split = 0;
  if (a.kv_splits > 1 && !kv_piece(a, t_lo, t_hi, split)) {  // under-filled launch, nothing left for this piece
    write_empty_partial_rows(a, w, wr, h, split);
    return;
  }

  // ---- pipeline: page ids run two tiles ahead, rows one tile ahead (in registers), LDS one
  // tile ahead of the MFMAs.  Loads past the last tile re-read the last tile.
  Stage<FP8> stg;
  PageIds<UNIFORM> pg;
  fetch_page_ids<UNIFORM>(pg, src, t_lo, tid);
  tile_gload<FP8, UNIFORM>(stg, src, a.kv, kh, vh, t_lo, tid, pg);
  fetch_page_ids<UNIFORM>(pg, src, t_lo + kBN, tid);
  tile_lstore<FP8>(stg, lds_k_buf[0], lds_v_buf[0], tid);
  tile_gload<FP8, UNIFORM>(stg, src, a.kv, kh, vh, t_lo + kBN, tid, pg);
  fetch_page_ids<UNIFORM>(pg, src, t_lo + 2 * kBN, tid);
  __syncthreads();
  int buf = 0;
  for (int tb = t_lo; tb < t_hi; tb += kBN, buf ^= 1) {
    const char* lds_k = lds_k_buf[buf];
    const char* lds_v = lds_v_buf[buf];
    uint64_t mask_word = 0;  // a caller's mask turned into bits by the pre-pass: one word per lane and tile
    if constexpr (EXT) {
      if (mc.mode == 1 && mc.bits) mask_word = mc.bits[min(tb >> 6, mc.bit_words - 1)];
    }
    if (tb + kBN < t_hi) {
      // the other buffer was last read before the barrier that ended the previous tile
      tile_lstore<FP8>(stg, lds_k_buf[buf ^ 1], lds_v_buf[buf ^ 1], tid);
      tile_gload<FP8, UNIFORM>(stg, src, a.kv, kh, vh, tb + 2 * kBN, tid, pg);
      fetch_page_ids<UNIFORM>(pg, src, tb + 3 * kBN, tid);
    }
    const bool vis = wr.active && (!causal || tb <= w.prefix + wr.r_hi) &&
                     (W_ <= 0 || tb + kBN - 1 > w.prefix + wr.r_lo - W_);
    if (vis) {
      const bool need_mask = (causal ? (tb + kBN - 1 > w.prefix + wr.r_lo) : (mc.mode == 1 || tb + kBN > w.kv_len)) ||
                             (W_ > 0 && tb <= w.prefix + wr.r_hi - W_);
      auto request = [&](auto tag, u32x4_t& to) __attribute__((always_inline)) {
        constexpr int f = decltype(tag)::value;
        if constexpr (f < 16) to = lds_ld16(lds_k + ((f & 1) * 32 + c) * kKPitch + h * 16 + (f >> 1) * 32);
        else to = lds_ld16(lds_v + ((f & 3) * 32 + c) * kVPitch + h * 16 + (((f >> 3) & 1) * 32 + ((f >> 2) & 1) * 16) * 2);
      };
      f32x16_t S[2];
      u32x4_t frag[EXT || !FP8 ? 1 : CAP ? 2 : UNIFORM ? 6 : 4];
      tile_scores(S, frag, qB, request);
      u32x4_t pB[2][2];
      softmax_tile<CAP, EXT>(S, O, m, l, sm, need_mask, tb, h, wr.qpos, W_, pB, mc, mask_word);
      tile_product(O, frag, pB, request);
    }
    __syncthreads();
  }
  if (a.kv_splits > 1) write_partial_rows(a, w, wr, O, l, h, m * sm.sc2, split);
  else write_rows(a, w, wr, O, l, h, m * sm.sc2);
}

}  // namespace

namespace {
// ---------------------------------------------------------------- custom masks as bits
// The caller's mask is one i32 per (query token, kv token).  Read where the scores are, a wave's 32 rows are 32
// separate 256-byte runs per tile -- four times the cache lines of the K/V tile itself, per query head.  This
// pre-pass reads it once, coalesced, and leaves one bit per pair (>= 1 keeps): bit t % 64 of word t / 64 of
// row `token`, mask_pitch words per row; tokens from kv_len on read as hidden.  grid = query tokens, 4 waves,
// wave w takes words w, w + 4, ...
__device__ __forceinline__ int mask_owner_of_token(const int32_t* cu_q_lens, int num_seqs, int tok) {
  int lo = 0, hi = num_seqs;  // last i with cu_q_lens[i] <= tok (zero-length sequences are skipped)
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cu_q_lens[mid] <= tok) lo = mid; else hi = mid;
  }
  return lo;
}

// grid = (query tokens, workgroups of a row, kMaskWords words at a time each); a wave has eight words, requested together.
// What bounds it: round trips to memory, so a workgroup has one for its words (all of a row in one workgroup, as it was first,
// were up to eight in a chain), and up to 63 sequences are searched, and where the row's words begin is worked out, in one.
// 6 verify steps of 4 tokens on 4421..15445 x 32 / 8 heads 112.4 -> 89.6 us (the call), 21 of 4 on 591..8700 122.3 -> 111.2, one of 8 on
// 16000 x 8 / 1 heads 50.5 -> 34.3.  Some 2048 workgroups at most: the bound on the lengths may be far above them, and those that find
// nothing are not free.
//
// A row of workgroups behind those (WRITE) puts the call's new tokens into the cache, one each: what finds a token's mask row
// finds its place in the cache too, and a launch of its own in front is spared: 4 of 16 tokens on 498..821 x 64 / 8 heads
// 24.9 -> 22.1 us, 30 of 8 on 100..2000 x 8 / 2 35.2 -> 31.4, 32 of 16 on 100..400 x 40 / 8 49.7 -> 46.0, the long contexts above
// 89.6 -> 85.9, 111.2 -> 107.1, 34.1 -> 31.2.
constexpr int kMaskWords = 32;
template <bool WRITE>
__global__ __launch_bounds__(256) void rpa_mask_bits_kernel(const PrefillArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // (masked calls run every sequence through the prefill kernels; with the composition on the device the number
  // of sequences is only a bound)
  int seq_end = a.seq_end, token, kv_len, width, seq, from_end;  // from_end: the sequence's tokens from this one on
  // where the sequence's rows start: given, or the sum over the sequences before it (cheap beside the rows themselves, and
  // the caller is spared a scan of its own)
  int64_t first = 0;
  if (seq_end < 64) {  // a sequence per lane
    const int s = min(lane, a.seq_end), own = min(lane, a.seq_end - 1);
    const int seqs_now = a.dist ? scalar_load_i32(a.dist + 2) : seq_end;
    const int q = a.pt.cu_q_lens[s], kv = a.pt.kv_lens[own];
    const int pages = a.sm.mask_rows_page_aligned ? a.pt.cu_kv_lens[s] : 0;
    const int given = a.sm.cu_mask_lens ? a.sm.cu_mask_lens[own] : 0;
    seq_end = max(min(seq_end, seqs_now), 0);
    token = __builtin_amdgcn_readlane(q, a.seq_begin) + (int)blockIdx.x;
    if (token >= __builtin_amdgcn_readlane(q, seq_end)) return;
    seq = max(__builtin_popcountll(__builtin_amdgcn_ballot_w64(lane < seq_end && q <= token)) - 1, 0);
    const int tokens = __shfl_down(q, 1) - q, row_width = a.sm.mask_rows_page_aligned ? __shfl_down(pages, 1) - pages : kv;
    kv_len = __builtin_amdgcn_readlane(kv, seq);
    width = __builtin_amdgcn_readlane(row_width, seq);
    from_end = __builtin_amdgcn_readlane(q, seq + 1) - token;
    if (a.sm.cu_mask_lens) {
      first = __builtin_amdgcn_readlane(given, seq);
    } else {
      first = lane < seq ? (int64_t)tokens * row_width : 0;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) first += __shfl_xor(first, off);
    }
    first += (int64_t)(token - __builtin_amdgcn_readlane(q, seq)) * width;
  } else {
    if (a.dist) seq_end = min(seq_end, a.dist[2]);
    token = a.pt.cu_q_lens[a.seq_begin] + (int)blockIdx.x;
    if (token >= a.pt.cu_q_lens[seq_end]) return;
    seq = mask_owner_of_token(a.pt.cu_q_lens, seq_end, token);
    from_end = a.pt.cu_q_lens[seq + 1] - token;
    kv_len = a.pt.kv_lens[seq];
    width = a.sm.mask_rows_page_aligned ? (a.pt.cu_kv_lens[seq + 1] - a.pt.cu_kv_lens[seq]) : kv_len;
    if (a.sm.cu_mask_lens) {
      first = a.sm.cu_mask_lens[seq];
    } else {
      for (int s = lane; s < seq; s += 64) {
        const int n = a.pt.cu_q_lens[s + 1] - a.pt.cu_q_lens[s];
        first += (int64_t)n * (a.sm.mask_rows_page_aligned ? a.pt.cu_kv_lens[s + 1] - a.pt.cu_kv_lens[s] : a.pt.kv_lens[s]);
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) first += __shfl_xor(first, off);
    }
    first += (int64_t)(token - a.pt.cu_q_lens[seq]) * width;
  }
  if (WRITE && blockIdx.y == gridDim.y - 1) {
    const KvWriteArgs& wr = a.write;
    const int pos = kv_len - from_end;
    if (pos < 0) return;
    const int slot = pos / wr.pt.page_size;
    const int page = wr.pt.page_indices[slot + (wr.pt.cu_kv_lens ? (int64_t)(wr.pt.cu_kv_lens[seq] / wr.pt.page_size)
                                                                 : (int64_t)seq * wr.pt.pages_per_seq)];
    const int64_t to = (int64_t)page * wr.kv.page_stride + (int64_t)(pos - slot * wr.pt.page_size) * wr.kv.tok_stride;
    const int pieces = wr.Hkv * wr.head_bytes / 16;
    for (int i = threadIdx.x; i < 2 * pieces; i += 256) {  // the key's, then the value's
      const bool value = i >= pieces;
      const int byte = (value ? i - pieces : i) * 16;
      const int head = byte / wr.head_bytes, inner = byte - head * wr.head_bytes;
      const bool real = inner < wr.src_head_bytes;  // (a narrow head's row ends in zeros)
      const char* from = (value ? wr.values : wr.keys) + ((int64_t)token * wr.Hkv + head) * wr.src_head_bytes + inner;
      st16(const_cast<char*>(value ? wr.kv.v_base : wr.kv.k_base) + to + (int64_t)head * wr.kv.head_stride + inner,
           real ? ld16(from) : u32x4_t{0u, 0u, 0u, 0u});
    }
    return;
  }
  const int32_t* row = a.sm.custom_mask + first;
  uint64_t* out = a.mask_bits + (int64_t)token * a.mask_pitch;
  const int words = min((kv_len + 63) >> 6, a.mask_pitch);
  for (int k0 = (int)blockIdx.y * kMaskWords + wave; k0 < words; k0 += ((int)gridDim.y - (WRITE ? 1 : 0)) * kMaskWords) {
    int v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int t = 64 * (k0 + 4 * i) + lane;
      v[i] = (t < kv_len) ? row[t] : 0;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint64_t keep = __ballot(v[i] >= 1);
      if (lane == 0 && k0 + 4 * i < words) out[k0 + 4 * i] = keep;
    }
  }
}

hipError_t launch_mask_bits(const PrefillArgs& a, hipStream_t stream) {
  if (!a.mask_bits || a.num_tokens <= 0) return hipSuccess;
  const int most = std::max(1, 2048 / a.num_tokens);
  const unsigned parts = (unsigned)std::min((a.mask_pitch + kMaskWords - 1) / kMaskWords, most);
  if (a.write.keys)
    hipLaunchKernelGGL((rpa_mask_bits_kernel<true>), dim3((unsigned)a.num_tokens, parts + 1), dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL((rpa_mask_bits_kernel<false>), dim3((unsigned)a.num_tokens, parts), dim3(256), 0, stream, a);
  return hipGetLastError();
}

bool takes_pipe_kernel(const PrefillArgs& a) { return prefill_shape(a).kernel == kKernelPrefillPipe; }
}  // namespace

namespace {
// The compiled flash kernels' short-chunk tile: 32 positions x 4 heads per workgroup (rows "prefill_options_short"
// and "prefill_fp8_short" of the shape table).  RPA_PREFILL_STAGED=1 (bf16 rows through the register-staged
// kernel, a testing path) has no such tile.
bool compiled_short_chunk_tile(const PrefillArgs& a) {
  if (tuning().prefill_staged == 1 && !a.fp8) return false;
  const ShapeRule& r = prefill_shape(a);
  return r.kernel != kKernelPrefillPipe && r.tile_q == 32;
}
}  // namespace

const ShapeRule& prefill_shape_of(const PrefillArgs& a) {
  // RPA_PREFILL_STAGED=1 on a bf16 cache is a testing path outside the table: the fp8 kernel's rows
  return prefill_shape(a);
}

int prefill_kv_splits(const PrefillArgs& a) {
  return a.packed ? a.packed : prefill_unpacked_kv_splits(a, nullptr);
}

int prefill_unpacked_kv_splits(const PrefillArgs& a, double* us) {
  const int nseq = a.seq_end - a.seq_begin;
  if (takes_pipe_kernel(a)) return prefill_pipe_kv_splits(a, nseq, us);
  // the compiled kernels: a tile takes about 0.85 us alone on its CU (e4m3 1.05, 256-wide heads 2.0)
  const bool heads4 = compiled_short_chunk_tile(a);
  return kv_pieces(a, nseq, heads4 ? 32 : kBM, heads4 ? 4 : 1, a.head_dim == 256 ? 2.0 : a.fp8 ? 1.05 : 0.85, us);
}

size_t prefill_split_workspace_bytes(const PrefillArgs& a, int splits) {
  return splits > 1 ? (size_t)a.num_tokens * a.Hq * splits * (a.head_dim + 2) * sizeof(float) : 0;
}

static int64_t compiled_grid(PrefillArgs& a, int nseq, bool heads4, int& tiles, bool& by_level) {
  const int bm = heads4 ? 32 : kBM;
  tiles = (a.max_q_len + bm - 1) / bm;
  // levels 0 .. ceil(max_kv_len / rows): only worth their empty workgroups when prefixes are
  // not much longer than the chunks (else every tile of a sequence costs about the same anyway)
  const bool level_order = tuning().prefill_level_order != 0;
  const int levels = a.max_kv_len > 0 ? (a.max_kv_len + bm - 1) / bm + 1 : 0;
  by_level = level_order && a.sm.mask_mode == 0 && levels > tiles && levels <= 2 * tiles + 2;
  if (by_level) tiles = levels;
  return prefill_grid(a, nseq, tiles, GridShape{bm, heads4 ? 4 : 1, a.head_dim == 256 ? 0 : 64, false});
}

bool prefill_by_streams(const PrefillArgs& call) {
  PrefillArgs a = call;
  const int nseq = a.seq_end - a.seq_begin;
  if (nseq <= 0 || a.max_q_len <= 0 || a.packed) return false;
  int tiles;
  bool by_level;
  if (takes_pipe_kernel(a)) prefill_pipe_grid(a, nseq, tuning().prefill_level_order != 0);
  else compiled_grid(a, nseq, compiled_short_chunk_tile(a), tiles, by_level);
  return a.map.block > 0;
}

hipError_t launch_prefill(const PrefillArgs& call, hipStream_t stream) {
  PrefillArgs a = call;
  const int nseq = a.seq_end - a.seq_begin;
  if (nseq <= 0 || a.max_q_len <= 0) return hipSuccess;
  if (a.packed) {
    if (a.sm.mask_mode == 1 && !a.mask_words) {
      hipError_t e = launch_mask_bits(a, stream);
      if (e != hipSuccess) return e;
    }
    return launch_prefill_packed(a, nseq, stream);
  }
  if (takes_pipe_kernel(a)) {
    return launch_prefill_pipe(a, nseq, tuning().prefill_level_order != 0, stream);
  }
  const bool heads4 = compiled_short_chunk_tile(a);
  int tiles;
  bool by_level;
  const int64_t grid = compiled_grid(a, nseq, heads4, tiles, by_level);
  if (grid + a.write_blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  // whether the rows that a wave brings in of a tile are one page's
  const int wave_rows = a.head_dim == 256 ? 8 : (a.fp8 || tuning().prefill_staged == 1) ? kBN : 16;
  const bool uniform = (a.pt.page_size % wave_rows) == 0;
  // soft cap and logit rounding share the general score path
  const bool cap = a.sm.soft_cap != 0.f || a.sm.round_logits != 0;
  const bool staged = a.fp8 || tuning().prefill_staged == 1;
  if (a.sm.mask_mode == 1) {
    hipError_t e = launch_mask_bits(a, stream);
    if (e != hipSuccess) return e;
  }
  const bool cut = a.kv_splits > 1;  // pieces of the K/V ranges on the second grid dimension, then the merge
  if (cut && (!a.ws_o || !a.ws_ml || a.kv_splits > 64)) return hipErrorInvalidValue;
  const dim3 g((unsigned)(grid + a.write_blocks), cut ? (unsigned)a.kv_splits : 1u), blk(256);
  const bool ext = a.sm.xai_len > 0.f || a.sm.mask_mode != 0 || a.sm.q_scale > 0.f;
#define RPA_STAGED(F, U, C, E) \
  hipLaunchKernelGGL((rpa_prefill_staged_kernel<F, U, C, E>), g, blk, 0, stream, a, tiles, nseq, by_level)
#define RPA_STAGED_FP8_HEADS4(U, C, E) \
  hipLaunchKernelGGL((rpa_prefill_staged_kernel<true, U, C, E, true>), g, blk, 0, stream, a, tiles, nseq, by_level)
#define RPA_ASYNC(U, C, E) hipLaunchKernelGGL((rpa_prefill_async_kernel<U, C, E>), g, blk, 0, stream, a, tiles, nseq, by_level)
#define RPA_ASYNC_HEADS4(U, C, E) \
  hipLaunchKernelGGL((rpa_prefill_async_kernel<U, C, E, true>), g, blk, 0, stream, a, tiles, nseq, by_level)
#define RPA_WIDE(F, U, C, E) \
  hipLaunchKernelGGL((rpa_prefill_async_kernel_wide<U, C, E, F>), g, dim3(512), 0, stream, a, tiles, nseq, by_level)
#define RPA_PICK(M, ...)                                            \
  switch ((uniform ? 4 : 0) | (cap ? 2 : 0) | (ext ? 1 : 0)) {        \
    case 0: M(__VA_ARGS__ false, false, false); break;              \
    case 1: M(__VA_ARGS__ false, false, true); break;               \
    case 2: M(__VA_ARGS__ false, true, false); break;               \
    case 3: M(__VA_ARGS__ false, true, true); break;                \
    case 4: M(__VA_ARGS__ true, false, false); break;               \
    case 5: M(__VA_ARGS__ true, false, true); break;                \
    case 6: M(__VA_ARGS__ true, true, false); break;                \
    default: M(__VA_ARGS__ true, true, true); break;                \
  }
#define RPA_WIDE_FP8(U, C, E) RPA_WIDE(true, U, C, E)
#define RPA_WIDE_BF16(U, C, E) RPA_WIDE(false, U, C, E)
#define RPA_STAGED_FP8(U, C, E) RPA_STAGED(true, U, C, E)
#define RPA_STAGED_BF16(U, C, E) RPA_STAGED(false, U, C, E)
  if (a.head_dim == 256) {
    if (a.fp8) {
      RPA_PICK(RPA_WIDE_FP8, )
    } else {
      RPA_PICK(RPA_WIDE_BF16, )
    }
  } else if (heads4 && a.fp8) {
    RPA_PICK(RPA_STAGED_FP8_HEADS4, )
  } else if (heads4) {
    RPA_PICK(RPA_ASYNC_HEADS4, )
  } else if (!staged) {
    RPA_PICK(RPA_ASYNC, )
  } else if (a.fp8) {
    RPA_PICK(RPA_STAGED_FP8, )
  } else {
    RPA_PICK(RPA_STAGED_BF16, )
  }
#undef RPA_STAGED_FP8
#undef RPA_STAGED_BF16
#undef RPA_PICK
#undef RPA_STAGED
#undef RPA_ASYNC
#undef RPA_ASYNC_HEADS4
#undef RPA_STAGED_FP8_HEADS4
#undef RPA_WIDE
#undef RPA_WIDE_FP8
#undef RPA_WIDE_BF16
  return cut ? launch_prefill_combine(a, stream) : hipGetLastError();
}

}  // namespace rpa
