// Pieces shared by the prefill kernels (rpa_prefill.hip, rpa_prefill_pipe.hip): work
// decomposition, tile geometry in LDS, the asynchronous global -> LDS tile copy, the online
// softmax of a 64-token tile and the final row write.
#pragma once

#include "rpa_common.h"
#include "rpa_kernels.h"
#include "rpa_shapes.h"
#include "rpa_tuning.h"

namespace rpa {
namespace pf {

constexpr int kBM = 128;  // query rows per workgroup
constexpr int kBN = 64;   // kv tokens per tile

// A tile of 128-wide heads in LDS: rows stay row-major and unpadded (256-wide heads have a kernel and a layout of their own)
constexpr int kHeadDim = 128;
constexpr int kRowB = kHeadDim * 2;      // one K or V row of a head, bf16
constexpr int kTileB = kBN * kRowB;      // 16 KiB
constexpr int kChunks = kHeadDim / 8;    // 16-byte chunks per row
constexpr int kSteps = kHeadDim / 16;    // k-steps of the first product
constexpr int kDimTiles = kHeadDim / 32; // 32-dim output tiles of the second product
constexpr int kCopies = kChunks / 4;     // copy instructions per wave, for K and for V
constexpr int kRowsPerCopy = 64 / kChunks;

__device__ __forceinline__ u32x4_t lds_ld16(const char* p) { return *reinterpret_cast<const u32x4_t*>(p); }
__device__ __forceinline__ void lds_st16(char* p, u32x4_t v) { *reinterpret_cast<u32x4_t*>(p) = v; }

typedef short s16x4_t __attribute__((ext_vector_type(4)));

// ds_read_b64_tr_b16: inside every block of 16 lanes, lane i receives
//   out[e] = M[(i >> 2) + 4e][i & 3],  e = 0..3,
// where M[r][0..3] are the four 16-bit elements at the address supplied by lane r of
// the block.  With lane r pointing at (token r >> 2, dims 4*(r & 3) ..) of a row-major
// tile, lane i ends up with dim i of four tokens: the k-contiguous MFMA operand.
__device__ __forceinline__ u32x2_t lds_tr16(const char* p) {
  typedef __attribute__((address_space(3))) s16x4_t* lds_ptr_t;
  const s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)(p));
  return __builtin_bit_cast(u32x2_t, v);
}

// token (inside a 64-token tile) that lands at LDS position 8*tg + i of a staged V^T row
__device__ __forceinline__ int vt_token(int tg, int i) {
  return (tg >> 1) * 16 + (i >> 2) * 8 + (tg & 1) * 4 + (i & 3);
}

struct TileSrc {
  const int32_t* pages;
  int32_t page_size;
  int32_t page_shift;
  int32_t last_tok;
};

__device__ __forceinline__ int page_slot(const TileSrc& s, int tok) {
  return s.page_shift >= 0 ? (tok >> s.page_shift) : (tok / s.page_size);
}

// Byte offset of token `tok` of the tile starting at `tb`.  UNIFORM (page_size % 64 == 0):
// the tile lies inside the page `page`.
template <bool UNIFORM>
__device__ __forceinline__ int64_t row_offset(const TileSrc& s, const KvAddr& kv, int tb, int tok, int page) {
  tok = min(tok, s.last_tok);
  if constexpr (UNIFORM) {
    const int page_tok0 = page_slot(s, tb) * s.page_size;  // wave-uniform
    return (int64_t)page * kv.page_stride + (int64_t)(tok - page_tok0) * kv.tok_stride;
  } else {
    return (int64_t)page * kv.page_stride + (int64_t)(tok - page_slot(s, tok) * s.page_size) * kv.tok_stride;
  }
}

// ------------------------------------------------------------------ work decomposition
// A unit is one (sequence, kv head): its G query heads and all their query tiles read the same K/V.  Hardware deals
// workgroup n to XCD n % 8, and inside an XCD to its four shader engines in turn, whatever they have left to do.  So
//   * the G heads of a (unit, tile) pair sit next to each other on one XCD (one L2); pairs go round the XCDs, tile by tile;
//   * the places of a sequence's pairs change with the tile.  A ragged sequence, which has
//     workgroups for its own length only, then meets every shader engine, and with fewer than 8 kv heads other XCDs too (with
//     8, 16, ... its kv heads stay on theirs).  Six chunks of 341 .. 1473 tokens x 16 / 8 heads of 256 dims, in the same places
//     for every tile, had left 4 workgroups to each of 112 CUs and 1 to 48: 262.6 -> 203.5 us.  7 prompts of 264 .. 1643
//     tokens x 8 / 2 heads 46.6 -> 37.1, 4 prompts of 484 ..
//     2368 x 16 / 8 heads 119 -> 87; odd numbers of sequences and 4 heads per kv head are where they were.
// Sequences with much to read take the order by streams instead (STREAMS, a.map.block; streams_in_turn()): a.map.block tiles of one
// sequence and kv head, as many as an XCD has places for with their heads, come one after the other, then those of the next sequence.
// They walk the same K/V side by side, which their XCD's L2 then fetches once; in the order of pairs four sequences share it, and
// once workgroups of different lengths have ended, four heads are all that still walk together.
// The most expensive query tiles are issued first, so that the last workgroups to start are short ones.  A causal tile costs
// what its last row sees: with a bound on kv_len from the host, tiles are ordered by level = tile index + ceil(prefix / tile
// rows), i.e. by that extent across sequences; without one, by position inside their own sequence.
struct Work {
  int seq, hk, head, q_start, qg0, q_len, kv_len, prefix;
  bool valid;
};

// n / d by a multiplication, for n < 2^31: scalar instructions, where a division is some 40 of the vector pipe, one after the
// other, in front of everything else that a workgroup does.
__device__ __forceinline__ int by(int n, const FastDiv& d) {
  return (int)((__umulhi((uint32_t)n, d.mul) + (uint32_t)n) >> d.shift);
}
inline FastDiv fast_div(int d) {
  FastDiv f;
  f.shift = 0;
  while (((int64_t)1 << f.shift) < d) ++f.shift;
  f.mul = (uint32_t)((((uint64_t)1 << 32) * (((uint64_t)1 << f.shift) - (uint64_t)d)) / (uint64_t)d + 1);
  return f;
}

// `heads` query heads of a kv head per workgroup (1, or 4 when the waves of a workgroup take a head each):
// Work.head is then the first of them.
template <bool STREAMS = false>
__device__ __forceinline__ Work decompose(const PrefillArgs& a, int tiles, int nseq, bool by_level, int bm = kBM,
                                          int heads = 1) {
  Work w;
  w.valid = false;
  const int units = nseq * a.Hkv;
  const int groups = a.G / heads;  // workgroups per (sequence, kv head, tile)
  const int span = a.map.apart ? 1 : groups, per_kv = a.map.apart ? groups : 1;  // workgroups of a kv head side by side; its places
  const int r = blockIdx.x >> 3, rg = by(r, a.map.groups);
  int tile_rev, si, gi;
  if (STREAMS && a.map.block > 0) {
    const int run = a.map.block, of_seq = (a.Hkv >> 3) * run;  // pairs of one kv head and round; of a sequence, on one XCD
    const int round = by(rg, a.map.round), in_round = rg - round * of_seq * nseq;
    si = by(in_round, a.map.seq_round);
    const int in_seq = in_round - si * of_seq, turn = by(in_seq, a.map.run);
    tile_rev = (round * run) + in_seq - turn * run;
    if (tile_rev >= tiles) return w;
    w.hk = turn * 8 + (blockIdx.x & 7);
    gi = (r - rg * span) * heads;
  } else {
    const int pair = rg * 8 + (blockIdx.x & 7);
    tile_rev = by(pair, a.map.units);
    if (tile_rev >= tiles) return w;
    const int place = pair - tile_rev * (units * per_kv);
    si = by(place, a.map.hkv);
    const int in_seq = place - si * (a.Hkv * per_kv);
    w.hk = by(in_seq, a.map.per_kv);
    gi = ((r - rg * span) + (in_seq - w.hk * per_kv)) * heads;
    if ((nseq & 1) == 0) {  // (an odd number of them moves on by itself)
      si += tile_rev;
      si -= by(si, a.map.nseq) * nseq;
    }
  }
  w.head = w.hk * a.G + gi;
  w.seq = a.seq_begin + si;
  if (w.seq >= a.seq_end) return w;  // the grid was sized for a bound on the number of sequences
  // (scalar loads, said explicitly here and below: in a kernel that also writes the cache the compiler takes no ordinary
  // load for one of memory that stays as it is, and fetches the lengths through the vector memory pipe)
  w.qg0 = scalar_load_i32(a.pt.cu_q_lens + w.seq);
  w.q_len = scalar_load_i32(a.pt.cu_q_lens + w.seq + 1) - w.qg0;
  w.kv_len = scalar_load_i32(a.pt.kv_lens + w.seq);
  w.prefix = w.kv_len - w.q_len;
  int tile = tiles - 1 - tile_rev;
  if (by_level) tile -= (max(w.prefix, 0) + bm - 1) / bm;
  w.q_start = tile * bm;
  if (tile < 0 || w.q_start >= w.q_len) return w;
  w.valid = true;
  return w;
}

// Whether a launch takes the order by streams (decompose): several sequences on a multiple of 8 kv heads with 4608 tokens or more to
// read for one of them, and the workgroups that have a tile, `work`, fit into the places at once or are 5/3 of them and more.  Known on
// the host and of the chunks themselves (behind decode rows the bound on the lengths may be theirs).
// What it gives is one K/V on its way to an XCD at a time, where four side by side do not stay in 4 MB, and long sequences that start first
// although they are few tiles.  What it costs is the end: the last sequence's workgroups start last, whatever they have to read, and
// where they are the few of a second round they are waited for.  In order of pairs -> by streams, us, prefixes ragged / all 5000 .. 6000:
//   fits         32 / 8 heads, 1905 + 60 tokens e4m3 323 -> 312, 40 / 8 heads, 1400 + 100 e4m3 371 -> 266 and bf16 283 -> 208
//   more         4 chunks of 1900 .. 2048 x 32 / 8 1500 -> 1382 (4.2 GB past the L2s for 0.2 GB of cache, now 0.35), 4 of 1000 bf16
//                571 -> 514 and e4m3 777 -> 680, with a cap 864 -> 750, 2 of 2400 x 24 / 8 648 -> 519 and e4m3 871 -> 698, 6 of 1500 x 16 / 8
//                446 -> 406 and e4m3 590 -> 495, 5 of 500 .. 3000 x 64 / 16 1318 -> 1249;
//                even prefixes are level, 0.97 .. 1.06; at worst 2400 on 3400 and 2300 on 13800 x 32 / 16 771 -> 816 (the longer first
//                781 -> 747), 1900 + 300 + 200 x 64 / 16 e4m3 648 -> 685
//   between      e4m3 1905 + 321 on 5811 375 -> 386, 1905 + 700 400 -> 439, 1500 + 900 386 -> 432, bf16 with a cap 394 -> 405, 3 of 2000 x 16 / 8
//                e4m3 382 -> 410; others gain (1905, 321, 400 e4m3 501 -> 474), and nothing that the host knows tells them apart.
//                The assembly kernel on four heads or more per kv head waits for the L2s most and does gain: 1905 + 321 bf16 309 -> 286,
//                1500 + 900 314 -> 286, 900 + 1905 328 -> 309, 64 / 8 900 + 100 297 -> 272, at worst 1905 + 1200 347 -> 351.
// On up to 4600 tokens the two orders are level or the order of pairs ahead (chunks of 29 .. 1946 on 276 58 against 61), and with 256-wide
// heads, one workgroup to a CU, 0.95 .. 1.0.  Fewer kv heads would spread a sequence over the XCDs by its tiles: 0.72 .. 1.28 times as
// fast, by how the tiles come out.  (The bound is one of tokens for both element types: e4m3 on 4000 .. 6000, 4 of 1000, 464 -> 448.)
struct GridShape {
  int bm, heads;  // query positions and heads of a workgroup
  int slots;      // workgroups that an XCD has places for, of a kernel that knows the order by streams (0: it does not)
  bool assembly;
};
inline bool streams_in_turn(const PrefillArgs& a, int nseq, int64_t grid, const GridShape& s) {
  if (s.slots <= 0 || nseq <= 1 || a.Hkv % 8 != 0 || a.dist || a.seq_begin != 0) return false;
  const int64_t seen = a.sm.window > 0 ? std::min<int64_t>(a.max_kv_len, (int64_t)a.sm.window + kBM) : a.max_kv_len;
  const int64_t places = 8ll * s.slots;
  if (seen < 4608 || grid <= places) return false;
  const int groups = a.G / s.heads;
  const int64_t work = ((int64_t)a.num_tokens + nseq * (s.bm / 2)) / s.bm * groups * a.Hkv;  // (a sequence's last tile is half full on average)
  return (s.assembly && groups >= 4) || work <= places || 3 * work >= 5 * places;
}

// Workgroups of a launch of `tiles` tiles, and the divisors of their order (see decompose).
// With fewer than 8 units their heads go to XCDs of their own: what few pairs there are would leave XCDs without work (2 chunks of
// 36 .. 171 tokens x 8 / 1 heads 42.8 -> 31.5 us).
inline int64_t prefill_grid(PrefillArgs& a, int nseq, int tiles, const GridShape& s) {
  const int groups = a.G / s.heads, units = nseq * a.Hkv;
  a.map.apart = units < 8;
  const int span = a.map.apart ? 1 : groups, per_kv = groups / span;
  a.map.groups = fast_div(span);
  a.map.units = fast_div(units * per_kv);
  a.map.hkv = fast_div(a.Hkv * per_kv);
  a.map.per_kv = fast_div(per_kv);
  a.map.nseq = fast_div(nseq);
  a.map.block = 0;
  const int64_t grid = ((int64_t)units * per_kv * tiles + 7) / 8 * 8 * span;
  if (streams_in_turn(a, nseq, grid, s)) {
    const int most = std::max(1, s.slots / groups), rounds = (tiles + most - 1) / most, m = a.Hkv / 8;
    a.map.block = (tiles + rounds - 1) / rounds;
    a.map.run = fast_div(a.map.block);
    a.map.seq_round = fast_div(a.map.block * m);
    a.map.round = fast_div(a.map.block * m * nseq);
    return (int64_t)8 * m * nseq * rounds * a.map.block * groups;
  }
  return grid;
}

// K (or V) rows of the workgroup's kv head, token 0 of its sequence's first page.
__device__ __forceinline__ const char* head_rows(const PrefillArgs& a, const Work& w, const char* base) {
  return base + (int64_t)w.hk * a.kv.head_stride + (a.rows_are_new ? (int64_t)w.qg0 * a.kv.tok_stride : 0);
}

// The workgroups behind those of the attention itself leave the new tokens in the cache: a wave takes a token at a time.
// The attention does not wait for them (it reads the caller's rows), and a launch in front of it is saved: 4.3 us of the 25
// that a prompt of 1003 tokens on 8 heads took.  Called by the workgroups that decompose() finds no tile for, as it does for
// those behind the attention's (a question in front of it is a load that every workgroup waits for: 2.5 us of the 317 of a
// mixed batch that writes nothing here).
__device__ __forceinline__ void write_new_tokens(const PrefillArgs& a) {
  const int first = (int)gridDim.x - a.write_blocks;
  if ((int)blockIdx.x < first || blockIdx.y != 0) return;
  const KvWriteArgs& wr = a.write;
  const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  const int t0 = ((int)blockIdx.x - first) * a.write_tokens;
  const int t1 = min(t0 + a.write_tokens, min(wr.num_tokens, scalar_load_i32(wr.pt.cu_q_lens + wr.num_seqs)));
  const int row_bytes = wr.Hkv * wr.head_bytes;
  for (int t = t0 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); t < t1; t += waves) {
    int lo = 0, hi = wr.num_seqs;  // last i with cu_q_lens[i] <= t
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (scalar_load_i32(wr.pt.cu_q_lens + mid) <= t) lo = mid; else hi = mid;
    }
    const int pos = t - scalar_load_i32(wr.pt.cu_q_lens + lo);  // (no prefix)
    const int slot = __builtin_amdgcn_readfirstlane(pos / wr.pt.page_size);
    const int page = scalar_load_i32(wr.pt.page_indices + slot +
                                     (wr.pt.cu_kv_lens ? (int64_t)(scalar_load_i32(wr.pt.cu_kv_lens + lo) / wr.pt.page_size)
                                                       : (int64_t)lo * wr.pt.pages_per_seq));
    const int64_t off = (int64_t)page * wr.kv.page_stride + (int64_t)(pos - slot * wr.pt.page_size) * wr.kv.tok_stride;
    const int64_t from = (int64_t)t * row_bytes;
    for (int b = lane * 16; b < row_bytes; b += 1024) {
      const int head = b / wr.head_bytes;
      const int64_t at = off + (int64_t)head * wr.kv.head_stride + (b - head * wr.head_bytes);
      st16(const_cast<char*>(wr.kv.k_base) + at, ld16(wr.keys + from + b));
      st16(const_cast<char*>(wr.kv.v_base) + at, ld16(wr.values + from + b));
    }
  }
}

// The same for sequences with a prefix, in front of which nothing wrote (a.tail_is_new).
__device__ __forceinline__ void write_tail_tokens(const PrefillArgs& a) {
  const int first = (int)gridDim.x - a.write_blocks;
  if ((int)blockIdx.x < first || blockIdx.y != 0) return;
  const KvWriteArgs& wr = a.write;
  const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  // A sequence per lane: whose a token is, and where its pages begin, in one trip to memory for up to 63 of them (looked up one after the
  // other, as before, these workgroups, the last to start, ended the launch: 0.5 us per trip and token).
  const bool few = wr.num_seqs < 64;
  int q = 0, kv = 0, first_page = 0;
  if (few) {
    const int s = min(lane, wr.num_seqs), own = min(lane, wr.num_seqs - 1);
    q = wr.pt.cu_q_lens[s];
    kv = wr.pt.kv_lens[own];
    first_page = wr.pt.cu_kv_lens ? wr.pt.cu_kv_lens[own] : 0;
  }
  const int t0 = ((int)blockIdx.x - first) * a.write_tokens;
  const int t1 = min(t0 + a.write_tokens, min(wr.num_tokens, few ? __builtin_amdgcn_readlane(q, wr.num_seqs) : scalar_load_i32(wr.pt.cu_q_lens + wr.num_seqs)));
  const int row_bytes = wr.Hkv * wr.head_bytes;
  for (int t = t0 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); t < t1; t += waves) {
    const int64_t from = (int64_t)t * row_bytes;
    u32x4_t k = {}, v = {};  // the row's first KiB: asked for before its place is known
    if (lane * 16 < row_bytes) {
      k = ld16(wr.keys + from + lane * 16);
      v = ld16(wr.values + from + lane * 16);
    }
    int seq, next, kv_len, page0;
    if (few) {
      seq = max(__builtin_popcountll(__builtin_amdgcn_ballot_w64(lane < wr.num_seqs && q <= t)) - 1, 0);
      next = __builtin_amdgcn_readlane(q, seq + 1);
      kv_len = __builtin_amdgcn_readlane(kv, seq);
      page0 = __builtin_amdgcn_readlane(first_page, seq);
    } else {
      int lo = 0, hi = wr.num_seqs;  // last i with cu_q_lens[i] <= t
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (scalar_load_i32(wr.pt.cu_q_lens + mid) <= t) lo = mid; else hi = mid;
      }
      seq = lo;
      next = scalar_load_i32(wr.pt.cu_q_lens + lo + 1);
      kv_len = scalar_load_i32(wr.pt.kv_lens + lo);
      page0 = wr.pt.cu_kv_lens ? scalar_load_i32(wr.pt.cu_kv_lens + lo) : 0;
    }
    const int pos = kv_len - (next - t);
    if (pos < 0) continue;
    const int slot = __builtin_amdgcn_readfirstlane(pos / wr.pt.page_size);
    const int page = scalar_load_i32(wr.pt.page_indices + slot + (wr.pt.cu_kv_lens ? (int64_t)__builtin_amdgcn_readfirstlane(page0 / wr.pt.page_size)
                                                                                   : (int64_t)seq * wr.pt.pages_per_seq));
    const int64_t off = (int64_t)page * wr.kv.page_stride + (int64_t)(pos - slot * wr.pt.page_size) * wr.kv.tok_stride;
    for (int b = lane * 16; b < row_bytes; b += 1024) {
      if (b >= 1024) {
        k = ld16(wr.keys + from + b);
        v = ld16(wr.values + from + b);
      }
      const int head = b / wr.head_bytes;
      const int64_t at = off + (int64_t)head * wr.kv.head_stride + (b - head * wr.head_bytes);
      st16(const_cast<char*>(wr.kv.k_base) + at, k);
      st16(const_cast<char*>(wr.kv.v_base) + at, v);
    }
  }
}

__device__ __forceinline__ TileSrc make_src(const PrefillArgs& a, const Work& w) {
  TileSrc src;
  src.page_size = a.pt.page_size;
  src.page_shift = ((src.page_size & (src.page_size - 1)) == 0) ? (31 - __builtin_clz(src.page_size)) : -1;
  src.last_tok = w.kv_len - 1;
  src.pages = a.pt.page_indices + (a.pt.cu_kv_lens ? (scalar_load_i32(a.pt.cu_kv_lens + w.seq) / a.pt.page_size)
                                                  : (int64_t)w.seq * a.pt.pages_per_seq);
  return src;
}

// ------------------------------------------------------------------ per-wave state and softmax
struct WaveRows {
  int r_lo, r_hi, row, qpos;
  bool active;
};

template <bool CAP>
struct Softmax {
  float scale, cap, inv_cap;
  float sc2;   // raw score -> log2 units inside the exponent (per row: carries the temperature factor)
  float temp;  // soft-cap path: temperature factor
  int round_mode;   // soft-cap path: logits rounded to bf16 (1) or f16 (2) before the softmax
};

// Online-softmax update of one 64-token tile.  On entry S holds raw scores (MFMA units); on
// exit it holds the probabilities.  Scores stay in MFMA units; sc2 turns them into log2 units
// inside the exponent: p = 2^(s*sc2 - m*sc2) is one fused multiply-add per score (soft-capped
// scores are already in log2 units, sc2 = 1).  The running max starts at a finite floor far
// above the mask value, so a row whose tokens are all masked in this tile gets p = 0, not 2^0.
constexpr f32x16_t kZero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
constexpr float kMaxFloor = -1.0e30f;
constexpr float kMaskRaw = -3.0e38f;

// The kernels that keep scores unscaled take the maximum over them, with masked ones far below: a scale has to be positive.  The
// sign of a negative one goes into the queries (exact); one of nothing makes every score zero (0 x q: a query that is infinite
// or no number stays no number).  A scale that is no number is left alone: it reaches every sum and every output.
template <int N>
__device__ __forceinline__ void make_scale_positive(float& scale, u32x4_t (&q)[N]) {
  if (!(scale <= 1e-25f)) return;
  const bool nothing = scale >= -1e-25f;
#pragma unroll
  for (int ks = 0; ks < N; ++ks)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t x = q[ks][e];
      const uint32_t lost = ((x & 0x7f80u) == 0x7f80u ? 0x7fc0u : 0u) | ((x & 0x7f800000u) == 0x7f800000u ? 0x7fc00000u : 0u);
      q[ks][e] = nothing ? lost : x ^ 0x80008000u;
    }
  scale = nothing ? 1.0f : -scale;
}

// The running max is allowed to go stale: it is raised (and the accumulators rescaled) only
// when some row's new maximum exceeds it by more than 2^kMaxSlack, so probabilities stay
// below 2^kMaxSlack -- harmless in f32 sums and bf16 operands -- and the 64-register rescale
// of O happens a handful of times per row instead of once per tile.
constexpr float kMaxSlack = 8.0f;

__device__ __forceinline__ void update_running_max(float mx, float& m, float& l, f32x16_t (&O)[kDimTiles], float sc2) {
  if (__builtin_amdgcn_ballot_w64((mx - m) * sc2 > kMaxSlack) != 0) {
    const float m_new = fmaxf(m, mx);
    const float alpha = fast_exp2((m - m_new) * sc2);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int d = 0; d < kDimTiles; ++d)
#pragma unroll
      for (int v = 0; v < 16; ++v) O[d][v] *= alpha;
  }
}

// Which tokens a query row may see.  mode 0: causal (token <= row position); mode 1: the
// caller's mask row (>= 1 keeps), mode 2: everything; modes 1 and 2 still hide the tokens of a
// partial last tile beyond kv_len.  The sliding window applies on top in every mode.
struct MaskCtx {
  int mode;
  int kv_len;
  const int32_t* row;    // mode 1: this lane's mask row (token t at row[t])
  const uint64_t* bits;  // mode 1: the same row as bits (token t = bit t % 64 of word t / 64), or nullptr
  int bit_words;         // words per bit row
};

__device__ __forceinline__ MaskCtx make_mask_ctx(const PrefillArgs& a, const Work& w, int row) {
  MaskCtx mc;
  mc.mode = a.sm.mask_mode;
  mc.kv_len = w.kv_len;
  mc.row = nullptr;
  mc.bits = nullptr;
  mc.bit_words = a.mask_pitch;
  if (mc.mode == 1 && a.mask_bits) mc.bits = a.mask_bits + (int64_t)(w.qg0 + min(row, w.q_len - 1)) * a.mask_pitch;
  if (mc.mode == 1 && a.sm.cu_mask_lens) {
    const int width = a.sm.mask_rows_page_aligned ? (a.pt.cu_kv_lens[w.seq + 1] - a.pt.cu_kv_lens[w.seq]) : w.kv_len;
    mc.row = a.sm.custom_mask + a.sm.cu_mask_lens[w.seq] + (int64_t)min(row, w.q_len - 1) * width;
  }
  return mc;
}

// mask_word: with a caller's mask turned into bits (mc.bits), the word of this tile's 64 tokens, which the
// caller fetches at the top of the tile's step, in FRONT of the next tile's copy: loads return in order, so
// the wait for it leaves the copy in flight.  Without the bits, one 4-byte load per score, here, behind the
// first product (which waits for the copy as well).
template <bool CAP, bool EXT>
__device__ __forceinline__ void softmax_tile(f32x16_t (&S)[2], f32x16_t (&O)[kDimTiles], float& m, float& l,
                                             const Softmax<CAP>& sm, bool need_mask, int tb, int h, int qpos,
                                             int window, u32x4_t (&pB)[2][2], const MaskCtx& mc,
                                             uint64_t mask_word = 0) {
  if constexpr (CAP) {
    if (sm.cap != 0.f && !sm.round_mode) {
      // soft cap alone (the usual case), constants folded: five instructions per score.
      // cap tanh(s scale / cap) temp log2e = k2 - 2 k2 / (2^(s k1) + 1)
      const float k1 = sm.scale * sm.inv_cap * (2.0f * kLog2e), k2 = sm.cap * sm.temp * kLog2e;
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          S[mt][v] = __builtin_fmaf(__builtin_amdgcn_rcpf(fast_exp2(S[mt][v] * k1) + 1.0f), -2.0f * k2, k2);
    } else {
      // the general path: soft cap (if any), temperature, then the logit rounded to the softmax dtype.  One loop
      // per combination, so that no score pays for a choice that is the same for the whole call.
      const bool capped = sm.cap != 0.f;
      const float k1 = sm.scale * sm.inv_cap * (2.0f * kLog2e), k2 = (capped ? sm.cap : sm.scale) * sm.temp;
      auto all_scores = [&](auto logit, auto rounded) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int v = 0; v < 16; ++v) S[mt][v] = rounded(logit(S[mt][v])) * kLog2e;
      };
      auto with_cap = [&](float s) { return __builtin_fmaf(__builtin_amdgcn_rcpf(fast_exp2(s * k1) + 1.0f), -2.0f * k2, k2); };
      auto no_cap = [&](float s) { return s * k2; };
      auto as_is = [](float x) { return x; };
      auto to_bf16 = [](float x) { return bf16_round(x); };
      auto to_f16 = [](float x) { return f16_round(x); };
      if (capped) {  // (rounded: the unrounded capped case is the branch above)
        if (sm.round_mode == 1) all_scores(with_cap, to_bf16);
        else all_scores(with_cap, to_f16);
      } else {
        if (sm.round_mode == 1) all_scores(no_cap, to_bf16);
        else if (sm.round_mode == 2) all_scores(no_cap, to_f16);
        else all_scores(no_cap, as_is);
      }
    }
  }
  if (EXT && need_mask && mc.mode == 1 && mc.bits) {
    // the caller's mask as bits: the tile's 64 tokens are one word, fetched by the caller at the top of the step
    const uint32_t half[2] = {(uint32_t)mask_word >> (4 * h), (uint32_t)(mask_word >> 32) >> (4 * h)};
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int tok = tb + mt * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
        bool masked = (tok >= mc.kv_len) || !((half[mt] >> (8 * (v >> 2) + (v & 3))) & 1u);
        masked = masked || (window > 0 && tok <= qpos - window);
        S[mt][v] = masked ? kMaskRaw : S[mt][v];
      }
  } else if (need_mask) {
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int tok = tb + mt * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
        bool masked;
        if (!EXT || mc.mode == 0) masked = tok > qpos;
        else masked = (tok >= mc.kv_len) || (mc.mode == 1 && mc.row[tok] < 1);
        masked = masked || (window > 0 && tok <= qpos - window);
        S[mt][v] = masked ? kMaskRaw : S[mt][v];
      }
  }
  // 32 scores -> 1 with three-operand maxima: 16 instructions instead of 31
  float mx = __builtin_fmaxf(__builtin_fmaxf(S[0][0], S[0][1]), S[1][0]);
#pragma unroll
  for (int v = 1; v < 16; ++v) {
    if (v < 15) mx = __builtin_fmaxf(__builtin_fmaxf(mx, S[0][v + 1]), S[1][v]);
    else mx = __builtin_fmaxf(mx, S[1][v]);
  }
  mx = swap_max(mx);
  update_running_max(mx, m, l, O, sm.sc2);
  const float neg_m = -m * sm.sc2;
  // probabilities go straight into bf16 pairs (the B operands of the second product); the row
  // sum is taken over the rounded pairs, one dot instruction per pair
  const bf16x2_t ones = {(__bf16)1.0f, (__bf16)1.0f};
  float ps0 = 0.f, ps1 = 0.f;
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      uint32_t w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float p0 = fast_exp2(__builtin_fmaf(S[mt][8 * kk + 2 * j], sm.sc2, neg_m));
        const float p1 = fast_exp2(__builtin_fmaf(S[mt][8 * kk + 2 * j + 1], sm.sc2, neg_m));
        w[j] = pack_bf16x2(p0, p1);
        if (j & 1) ps1 = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w[j]), ones, ps1, false);
        else ps0 = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w[j]), ones, ps0, false);
      }
      pB[mt][kk] = u32x4_t{w[0], w[1], w[2], w[3]};
    }
  l += ps0 + ps1;
}

// lane (c, h) holds query row c, dims 32d + 8*(v/4) + 4h + v%4 in O[d][v].  Stored from there a row got 16 bytes at a time; a lane that
// has no row of its own takes part in the exchange (row_of_32).  8 prompts of 500..1500 tokens x 32 / 8 heads 108.7 -> 102.0 us, 30 of
// 100..300 65.5 -> 60.9, 20 of 200..600 x 16 / 8 with a window and sinks 56.5 -> 52.2, 6 chunks of 200..900 e4m3 64.7 -> 61.9, the mixed batch of 56
// rows and 8 chunks 332 -> 325, 256-wide prompts 105 -> 101.  (Partial rows, 32 bytes at a time, lost 1 % by the exchange.)
template <int N = kDimTiles>
__device__ __forceinline__ void write_rows(const PrefillArgs& a, const Work& w, const WaveRows& wr, const f32x16_t (&O)[N], float l, int h, float m2) {
  l = swap_sum(l);
  if (!wr.active) return;
  const float vs = a.v_scale ? scalar_load_f32(a.v_scale + w.hk) : 1.0f;
  const float inv = a.sm.sink ? vs * sink_inverse(m2, l, sink_logit(a.sm.sink, a.sm.round_logits, w.head)) : vs / l;
  const int lane = threadIdx.x & 63, row = wr.r_lo + (lane & 15), dim = row_of_32_at(lane) / 2;
  uint16_t* op = a.out + ((int64_t)(w.qg0 + row) * a.Hq + w.head) * a.q_dim + dim;
  const int64_t upper_rows = (int64_t)16 * a.Hq * a.q_dim;
  const bool has_lower = row < w.q_len, has_upper = row + 16 < w.q_len;
#pragma unroll
  for (int d = 0; d < N; ++d) {
    u32x2_t p[4];
#pragma unroll
    for (int vq = 0; vq < 4; ++vq)
      p[vq] = u32x2_t{pack_bf16x2(O[d][4 * vq + 0] * inv, O[d][4 * vq + 1] * inv),
                      pack_bf16x2(O[d][4 * vq + 2] * inv, O[d][4 * vq + 3] * inv)};
    u32x4_t lower, upper;
    row_of_32(p, lower, upper);
    if (d * 32 + dim >= a.q_dim) continue;  // (narrow heads)
    if (has_lower) st16(op + d * 32, lower);
    if (has_upper) st16(op + d * 32 + upper_rows, upper);
  }
}

// -------------------------------------------------- the launch shape of a prefill call (rpa_shapes.h)
// RPA_PREFILL_PIPE=0 / RPA_PREFILL_STAGED=1 take the assembly kernel out of the selection, RPA_PREFILL_PIPE_TILE
// = 32 | 128 and RPA_PREFILL_PIPE_NQ=2 decide the short-chunk question by hand.
inline ShapeKey prefill_shape_key(const PrefillArgs& a) {
  const Tuning& tune = tuning();
  ShapeKey k = {};
  k.stage = kStagePrefill;
  k.kv_bits = a.fp8 ? 8 : 16;
  k.head_dim = a.head_dim;
  k.heads = a.G;
  k.max_q_len = a.max_q_len;
  if (tune.prefill_pipe_tile == 32) k.max_q_len = 1;
  else if (tune.prefill_pipe_tile != 0 || tune.prefill_pipe_nq == 2) k.max_q_len = 0;
  k.options = ((a.sm.soft_cap != 0.f || a.sm.round_logits != 0) ? kOptSoftCap : 0u) |
              (a.sm.mask_mode != 0 ? kOptMaskOther : 0u) | (a.sm.xai_len > 0.f ? kOptTemperature : 0u) |
              (a.sm.q_scale > 0.f ? kOptQScale : 0u) | a.page_options;
  return k;
}

inline const ShapeRule& prefill_shape(const PrefillArgs& a) {
  const Tuning& tune = tuning();
  const unsigned skip = (tune.prefill_pipe == 0 || tune.prefill_staged == 1) ? (1u << kKernelPrefillPipe) : 0u;
  return select_shape(prefill_shape_key(a), skip);
}

// -------------------------------------------------- K/V ranges cut into pieces (under-filled launches)
// A launch with far fewer workgroups than CUs (one long prompt on a few heads, a chunk on a long prefix, a
// verify step on a long context) cuts every workgroup's run of K/V tiles into a.kv_splits pieces; blockIdx.y
// picks the piece, which leaves its rows as they stand -- unnormalised accumulators, (reference, sum) of the
// probabilities in log2 units -- in workspace slot ((token, head), piece), and rpa_prefill_combine_kernel
// finishes them.
constexpr float kNoReference = -1.0e30f;  // reference of a row that met no visible token: weighs nothing in the merge

// The piece of [t_lo, t_hi) that this workgroup runs; false when nothing is left for it.
__device__ __forceinline__ bool kv_piece(const PrefillArgs& a, int& t_lo, int& t_hi, int& split) {
  split = blockIdx.y;
  const int nT = (t_hi - t_lo + kBN - 1) / kBN;
  // The host chose the number of pieces for the longest range it knew a bound of; a shorter range is cut into
  // fewer (no piece under four tiles), the workgroups of the others leave rows that weigh nothing.
  const int pieces = max(1, min(a.kv_splits, nT >> 2));
  // (the division runs on the vector pipe: say that its result is the same in every lane)
  const int per = __builtin_amdgcn_readfirstlane((nT + pieces - 1) / pieces);
  const int lo = split * per, hi = min(nT, lo + per);
  if (lo >= hi) return false;
  t_hi = min(t_hi, t_lo + hi * kBN);
  t_lo += lo * kBN;
  return true;
}

// lane (c, h) holds query row c, dims 32d + 8*(v/4) + 4h + v%4 in O[d][v]
// (of narrow heads the first N tiles of 32; the merge's sums of the others are not used)
template <int N = kDimTiles>
__device__ __forceinline__ void write_partial_rows(const PrefillArgs& a, const Work& w, const WaveRows& wr, const f32x16_t (&O)[N], float l, int h, float m2, int split) {
  typedef float f32x4_t __attribute__((ext_vector_type(4)));
  l += __shfl_xor(l, 32);
  if (!wr.active || wr.row >= w.q_len) return;
  const int64_t slot = ((int64_t)(w.qg0 + wr.row) * a.Hq + w.head) * a.kv_splits + split;
  float* op = a.ws_o + slot * kHeadDim + 4 * h;
#pragma unroll
  for (int d = 0; d < N; ++d)
#pragma unroll
    for (int vq = 0; vq < 4; ++vq)
      *reinterpret_cast<f32x4_t*>(op + d * 32 + vq * 8) =
          f32x4_t{O[d][4 * vq + 0], O[d][4 * vq + 1], O[d][4 * vq + 2], O[d][4 * vq + 3]};
  if (h == 0) {
    a.ws_ml[slot * 2] = fmaxf(m2, kNoReference);
    a.ws_ml[slot * 2 + 1] = l;
  }
}

template <int N = kDimTiles>
__device__ __forceinline__ void write_empty_partial_rows(const PrefillArgs& a, const Work& w, const WaveRows& wr, int h,
                                                         int split) {
  f32x16_t zero[N];
#pragma unroll
  for (int d = 0; d < N; ++d) zero[d] = kZero16;
  write_partial_rows(a, w, wr, zero, 0.f, h, kNoReference, split);
}

// Merge the kv_splits partial rows of one (query token, query head): out = sum_j O_j 2^(m_j - m*) /
// sum_j l_j 2^(m_j - m*).  grid = (tokens, Hq); one wave, HD / 64 dims per lane; lane j fetches (m_j, l_j).
template <int HD>
static __global__ __launch_bounds__(64) void rpa_prefill_combine_kernel(const PrefillArgs a) {
  constexpr int kDpl = HD / 64;
  typedef float fvec_t __attribute__((ext_vector_type(kDpl)));
  // (with the call's composition on the device the sequences to process are read there, as in the kernels)
  int seq_begin = a.seq_begin, seq_end = a.seq_end;
  if (a.dist) {
    seq_begin = (a.sm.mask_mode == 1) ? 0 : scalar_load_i32(a.dist);
    seq_end = min(seq_end, scalar_load_i32(a.dist + 2));
  }
  const int tok0 = scalar_load_i32(a.pt.cu_q_lens + seq_begin);
  const int tok1 = scalar_load_i32(a.pt.cu_q_lens + seq_end);
  const int token = tok0 + (int)blockIdx.x;
  if (token >= tok1) return;
  const int head = blockIdx.y, lane = threadIdx.x, n = a.kv_splits;
  const int64_t base = ((int64_t)token * a.Hq + head) * n;
  float mj = -INFINITY, lj = 0.f;
  if (lane < n) {
    mj = a.ws_ml[(base + lane) * 2];
    lj = a.ws_ml[(base + lane) * 2 + 1];
  }
  float mstar = mj;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mstar = fmaxf(mstar, __shfl_xor(mstar, off));
  const float wj = (lane < n) ? fast_exp2(mj - mstar) : 0.f;
  float den = lj * wj;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) den += __shfl_xor(den, off);
  float acc[kDpl];
#pragma unroll
  for (int e = 0; e < kDpl; ++e) acc[e] = 0.f;
  for (int j0 = 0; j0 < n; j0 += 8) {  // eight partial rows requested at a time
    fvec_t o[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      o[u] = *reinterpret_cast<const fvec_t*>(a.ws_o + (base + min(j0 + u, n - 1)) * HD + kDpl * lane);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float wu = (j0 + u < n) ? __shfl(wj, j0 + u) : 0.f;  // the repeated last row does not count
#pragma unroll
      for (int e = 0; e < kDpl; ++e) acc[e] += o[u][e] * wu;
    }
  }
  const float vs = a.v_scale ? a.v_scale[head / a.G] : 1.0f;
  const float inv = a.sm.sink ? vs * sink_inverse(mstar, den, sink_logit(a.sm.sink, a.sm.round_logits, head)) : vs / den;
  if (kDpl * lane >= a.q_dim) return;
  uint32_t* op = reinterpret_cast<uint32_t*>(a.out + ((int64_t)token * a.Hq + head) * a.q_dim + kDpl * lane);
#pragma unroll
  for (int e = 0; e < kDpl; e += 2) op[e / 2] = pack_bf16x2(acc[e] * inv, acc[e + 1] * inv);
}

inline hipError_t launch_prefill_combine(const PrefillArgs& a, hipStream_t stream) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t tokens = std::max<int64_t>(1, (int64_t)a.num_tokens - a.seq_begin);  // decode rows hold one token each
  const dim3 g((unsigned)tokens, (unsigned)a.Hq);
  if (a.head_dim == 256) hipLaunchKernelGGL(rpa_prefill_combine_kernel<256>, g, dim3(64), 0, stream, a);
  else hipLaunchKernelGGL(rpa_prefill_combine_kernel<128>, g, dim3(64), 0, stream, a);
  return hipGetLastError();
}

// How many pieces (1 = whole ranges): the count that minimises a small model of the launch, fitted to
// measurements of the pipelined kernel.  The critical path is the longest range, chain / n tiles per piece; a
// tile takes ~tile_us while every workgroup has a CU to itself (up to ~192 workgroups: the dispatcher does
// not spread them perfectly), 2.6 x that once two share every CU (512), in proportion in between, and the
// launch runs in rounds of 512 workgroups beyond; the merge costs a launch (~1.5 us) plus the partial rows'
// way to memory and back (~0.29 ns per (token, head, piece) of 128 dims).  A cut must save at least 2 us,
// leaves no piece under four tiles and makes at most 64 pieces.  bm / heads: query positions and query heads
// per workgroup.  RPA_PREFILL_SPLITS: 0 / 1 never, n forces n.
inline int kv_pieces(const PrefillArgs& a, int nseq, int bm, int heads, double tile_us, double* us_of_best = nullptr) {
  // (with the composition on the device nseq, max_q_len, max_kv_len and num_tokens are bounds: a launch that is
  // under-filled even by its bounds is cut, and every workgroup fits the piece count to its own range)
  if (nseq <= 0 || a.max_q_len <= 0 || a.max_kv_len <= 0 || a.num_tokens <= 0) return 1;
  const int forced = us_of_best ? -1 : tuning().prefill_splits;  // (who asks for the time asks for the model's plan)
  if (forced == 0 || forced == 1) return 1;
  if (forced > 1) return std::min(forced, 64);
  const int64_t tokens = std::max<int64_t>(1, (int64_t)a.num_tokens - a.seq_begin);
  const int64_t blocks = std::min<int64_t>((int64_t)nseq * ((a.max_q_len + bm - 1) / bm), tokens / bm + nseq);
  const int64_t wgs = blocks * a.Hkv * (a.G / heads);
  int64_t longest = a.max_kv_len;  // tokens of the longest range
  if (a.sm.window > 0) longest = std::min<int64_t>(longest, (int64_t)a.sm.window + bm + kBN);
  const int64_t chain = (longest + kBN - 1) / kBN;
  const int64_t cap = std::min<int64_t>(64, chain / 4);
  const double per_piece = 0.29e-3 * (double)tokens * a.Hq * (a.head_dim / 128);  // us per piece for the partial rows
  auto launch_us = [&](int n) {
    const double w = (double)wgs * n;
    const double rate = w <= 192 ? 1.0 : w <= 512 ? 1.0 + (w - 192) * (1.6 / 320) : 2.6 * (w / 512);
    return tile_us * rate * chain / n + (n > 1 ? 1.5 + per_piece * n : 0.0);
  };
  // (and the partial rows stay under 256 MB)
  const int64_t row_bytes = (int64_t)a.num_tokens * a.Hq * (a.head_dim + 2) * 4;
  const int64_t cap_ws = row_bytes > 0 ? ((int64_t)256 << 20) / row_bytes : 64;
  int best = 1;
  double best_us = launch_us(1) - 2.0;
  for (int n = 2; n <= cap && n <= cap_ws; ++n) {
    const double us = launch_us(n);
    if (us < best_us) {
      best_us = us;
      best = n;
    }
  }
  if (us_of_best) {
    // (for the time and not only the choice: workgroups beyond one per CU cost what a mean range costs, not the longest)
    const double mean = std::min<double>(longest, std::max(1.0, a.max_kv_len - 0.5 * (a.max_q_len - 1))) / longest;
    const double w = (double)wgs * best, rate = w <= 192 ? 1.0 : w <= 512 ? 1.0 + (w - 192) * (1.6 / 320) : 2.6 * (w / 512);
    *us_of_best = tile_us * chain / best * std::max(1.0, rate * mean * 1.15) + (best > 1 ? 1.5 + per_piece * best : 0.0);
  }
  return best;
}

// ==================================================================== async path (bf16 cache)
// 16-byte chunk j of row t sits at chunk position j ^ swizzle(t):
//   K: swizzle = t & 15      (ds_read_b128: 16 consecutive tokens -> 16 distinct chunk columns)
//   V: swizzle = 4 * (t & 3) (transposing read: 4 consecutive tokens -> 4 distinct 64-byte windows)
// Every wave copies kCopies x 64 chunks of K and of V: chunk position p = 64*(kCopies*wave + n) +
// lane of the tile, i.e. row p / kChunks, chunk column p % kChunks.
// Pages that hold whole groups of the ROWS consecutive rows that a wave copies of a tile (N copy instructions for K, N for V): one
// page id per wave and tile, a scalar base, and per lane offsets that never change.  An address per lane and copy -- 64-bit
// products, and ids through the vector memory pipe for pages under a tile -- was most of what a wave issued beside its matrix
// instructions.  Issued as assembly: the caller waits for the copies (vmcnt) itself.
template <int ROWS, int N>
struct RowFeed {
  uint32_t k[N], v[N];  // byte offset of this lane's chunk from the wave's first row
  int first, id;        // of the tile asked for last: the first row that the wave copies, and its page

  // `row(n)`: this lane's row of copy n, from the wave's first; chunk_k / chunk_v(n): the chunk that it moves
  template <class Row, class ChunkK, class ChunkV>
  __device__ __forceinline__ void init(const KvAddr& kv, Row row, ChunkK chunk_k, ChunkV chunk_v) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      k[n] = (uint32_t)(row(n) * kv.tok_stride + (chunk_k(n) << 4));
      v[n] = (uint32_t)(row(n) * kv.tok_stride + (chunk_v(n) << 4));
    }
  }
  // rows wave * ROWS .. of the tile at `tb`; past the end: the last rows again
  __device__ __forceinline__ void fetch_page(const TileSrc& s, int tb, int wave) {
    first = __builtin_amdgcn_readfirstlane(min(tb + wave * ROWS, s.last_tok & ~(ROWS - 1)));
    id = scalar_load_i32(s.pages + __builtin_amdgcn_readfirstlane(page_slot(s, first)));
  }
  __device__ __forceinline__ int64_t base(const TileSrc& s, const KvAddr& kv) const {
    return (int64_t)id * kv.page_stride + (int64_t)(first - page_slot(s, first) * s.page_size) * kv.tok_stride;
  }
  // `at`: LDS address of the wave's first KiB; `b`: the head's rows plus base()
  template <bool IS_V, class Row>
  __device__ __forceinline__ void copy(uint32_t at, const char* b, const TileSrc& s, const KvAddr& kv, Row row) const {
    if (first + ROWS - 1 <= s.last_tok) {
#pragma unroll
      for (int n = 0; n < N; ++n)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :: "s"(at + n * 1024), "v"(IS_V ? v[n] : k[n]), "s"(b) : "memory", "m0");
    } else {  // the sequence's last rows: those past its end repeat the last one
      const int last = s.last_tok - first;
#pragma unroll
      for (int n = 0; n < N; ++n) {
        const uint32_t o = (IS_V ? v[n] : k[n]) - (uint32_t)(max(row(n) - last, 0) * kv.tok_stride);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(at + n * 1024), "v"(o), "s"(b) : "memory", "m0");
      }
    }
  }
};

// Other page sizes: an address per lane and copy, from the page of the lane's row.
struct AsyncPages {
  int32_t id[kCopies];
};

__device__ __forceinline__ void async_fetch_pages(AsyncPages& pg, const TileSrc& s, int tb, int wave, int lane) {
  tb = min(tb, s.last_tok & ~(kBN - 1));
#pragma unroll
  for (int n = 0; n < kCopies; ++n) {
    const int t = (wave * kCopies + n) * kRowsPerCopy + lane / kChunks;
    pg.id[n] = s.pages[page_slot(s, min(tb + t, s.last_tok))];
  }
}

__device__ __forceinline__ void async_copy_tile(char* lds_k, char* lds_v, const TileSrc& s, const KvAddr& kv, const char* kh,
                                                const char* vh, int tb, int wave, int lane, const AsyncPages& pg) {
  typedef const __attribute__((address_space(1))) void* gptr_t;
  typedef __attribute__((address_space(3))) void* lptr_t;
  tb = min(tb, s.last_tok & ~(kBN - 1));  // past the end: re-copy the last tile
  const int cp = lane % kChunks;
#pragma unroll
  for (int n = 0; n < kCopies; ++n) {
    const int blk = wave * kCopies + n;
    const int t = blk * kRowsPerCopy + lane / kChunks;
    const int64_t ro = row_offset<false>(s, kv, tb, tb + t, pg.id[n]);
    const int jk = cp ^ (t & 15);
    const int jv = cp ^ ((t & 3) << 2);
    __builtin_amdgcn_global_load_lds((gptr_t)(kh + ro + jk * 16), (lptr_t)(lds_k + blk * 1024), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((gptr_t)(vh + ro + jv * 16), (lptr_t)(lds_v + blk * 1024), 16, 0, 0);
  }
}
}  // namespace pf

// rpa_prefill_pipe.hip: the software-pipelined kernel for the plain causal bf16 case
bool prefill_pipe_applies(const PrefillArgs& a);
hipError_t launch_prefill_pipe(const PrefillArgs& a, int nseq, bool level_order, hipStream_t stream);
// What the pipelined kernel is launched as; sets a.map.
struct PipeGrid {
  int nq, tiles;
  bool heads4, by_level;
  int64_t grid;
};
PipeGrid prefill_pipe_grid(PrefillArgs& a, int nseq, bool level_order);
int prefill_pipe_kv_splits(const PrefillArgs& a, int nseq, double* us = nullptr);

// rpa_prefill_packed.hip: 32 (position, head) columns per workgroup, whose waves walk different tiles
hipError_t launch_prefill_packed(const PrefillArgs& a, int nseq, hipStream_t stream);
// pieces of the other kernels and, in *us, what kv_pieces() gives their launch
int prefill_unpacked_kv_splits(const PrefillArgs& a, double* us);

}  // namespace rpa
