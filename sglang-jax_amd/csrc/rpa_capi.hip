// C ABI of the library (declared in include/rpa.h): argument checking,
// grid sizing from the host-side bounds, and dispatch to the kernel launchers.
// No device allocation, no synchronisation, no host reads of device memory.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstddef>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "../../include/rpa.h"
#include "rpa_kernels.h"
#include "rpa_tuning.h"

extern char** environ;

namespace rpa {

// One parse of the RPA_* switches per change of the environment (per thread), one look at it per call: see rpa_tuning.h.
static thread_local int g_calls = 0;        // entry points that this thread is in
static thread_local bool g_looked = false;  // inside them: the environment has been looked at
TuningOfCall::TuningOfCall() {
  if (g_calls++ == 0) g_looked = false;
}
TuningOfCall::~TuningOfCall() { --g_calls; }

const Tuning& tuning() {
  thread_local Tuning t;
  thread_local uint64_t seen = 0;
  thread_local bool valid = false;
  if (g_calls > 0) {
    if (g_looked) return t;
    g_looked = true;
  }
  // setenv() never edits a string in place: a changed variable is a changed pointer in environ
  uint64_t h = 1469598103934665603ull;
  for (char** e = environ; e && *e; ++e) h = (h ^ reinterpret_cast<uintptr_t>(*e)) * 1099511628211ull;
  if (valid && h == seen) return t;
  t = Tuning();
  auto geti = [](const char* name, int& dst) {
    const char* v = getenv(name);
    if (v && *v) dst = atoi(v);
  };
  geti("RPA_DECODE_MIN_CHUNK", t.decode_min_chunk);
  geti("RPA_DECODE_BALANCED", t.decode_balanced);
  geti("RPA_DECODE_WAVES_PER_WG", t.decode_waves_per_wg);
  geti("RPA_DECODE_WAVE_CAPACITY", t.decode_wave_capacity);
  geti("RPA_DECODE_ROW_KB", t.decode_row_kb);
  geti("RPA_DECODE_ROW_PIECES", t.decode_row_pieces);
  geti("RPA_DECODE_MERGE_IN_KERNEL", t.decode_merge_in_kernel);
  geti("RPA_DECODE_LDS_KB", t.decode_lds_kb);
  geti("RPA_MASK_BITS", t.mask_bits);
  geti("RPA_PREFILL_ROWS256", t.prefill_rows256);
  geti("RPA_PREFILL_STAGED", t.prefill_staged);
  geti("RPA_PREFILL_PIPE", t.prefill_pipe);
  geti("RPA_PREFILL_PIPE_TILE", t.prefill_pipe_tile);
  geti("RPA_PREFILL_LEVEL_ORDER", t.prefill_level_order);
  geti("RPA_PREFILL_PIPE_NQ", t.prefill_pipe_nq);
  geti("RPA_PREFILL_PIPE_MASKED", t.prefill_pipe_masked);
  geti("RPA_PREFILL_SPLITS", t.prefill_splits);
  geti("RPA_PREFILL_PACKED", t.prefill_packed);
  geti("RPA_MLA_MIN_CHUNK", t.mla_min_chunk);
  geti("RPA_MLA_WG_CAPACITY", t.mla_wg_capacity);
  geti("RPA_MLA_BALANCED", t.mla_balanced);
  geti("RPA_MLA_PIECE_PAD", t.mla_piece_pad);
  geti("RPA_MLA_PIPE", t.mla_pipe);
  geti("RPA_MLA_SHARED_TILES", t.mla_shared_tiles);
  geti("RPA_MLA_WIDE", t.mla_wide);
  geti("RPA_MLA_TOKEN_GROUPS", t.mla_token_groups);
  geti("RPA_MLA_WAVES", t.mla_waves);
  if (const char* v = getenv("RPA_PREFILL_PIPE_LIMIT")) {
    if (*v) t.prefill_pipe_limit = (float)atof(v);
  }
  seen = h;
  valid = true;
  return t;
}

int compute_units() {
  static const int n = [] {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) return v;
    return 256;
  }();
  return n;
}

}  // namespace rpa

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

// Held while a call's launches are enqueued: several threads may share a stream and with it a workspace, and between the
// launch that leaves partial rows there and the one that merges them no other call's may come.
class WorkspaceTurn {
 public:
  explicit WorkspaceTurn(const void* workspace) {
    static std::mutex turns[16];
    if (workspace) lock_ = std::unique_lock<std::mutex>(turns[(reinterpret_cast<uintptr_t>(workspace) >> 9) & 15]);
  }

 private:
  std::unique_lock<std::mutex> lock_;
};

constexpr float kDefaultMask = -0.7f * 3.4028234663852886e38f;

// Bytes of a custom mask as one bit per pair; 0: the kernels read the caller's i32 words (no bound on the lengths, 256-wide
// heads, a batch too large, RPA_MASK_BITS=0).
size_t mask_bits_bytes(const RpaParams* p) {
  if (p->mask_mode != RPA_MASK_CUSTOM || p->head_dim != 128 || p->max_kv_len <= 0 || p->num_tokens <= 0 || rpa::tuning().mask_bits == 0)
    return 0;
  const size_t bytes = (size_t)p->num_tokens * ((p->max_kv_len + 63) / 64) * sizeof(uint64_t);
  return bytes > ((size_t)256 << 20) ? 0 : bytes;
}
bool mask_as_bits(const RpaParams* p) { return mask_bits_bytes(p) != 0; }

// A caller's parameters as this build knows them.  The fields behind `distribution` came later: a caller compiled against
// an earlier header passes a struct that ends there, and nothing behind that is read unless `layout` says it is (rpa.h).
// Every entry point starts with one of these and works on its copy.
struct OwnParams {
  const rpa::TuningOfCall tuning;
  RpaParams own = {};
  const RpaParams* p = nullptr;  // nullptr where the caller's is
  explicit OwnParams(const RpaParams* given) {
    if (!given) return;
    const bool tail = given->layout == (RPA_LAYOUT_FUSED | RPA_PARAMS_TAIL) || given->layout == (RPA_LAYOUT_SPLIT | RPA_PARAMS_TAIL);
    memcpy(&own, given, tail ? sizeof(own) : offsetof(RpaParams, q_head_dim));
    if (own.layout == RPA_LAYOUT_FUSED || own.layout == RPA_LAYOUT_SPLIT) own.layout |= RPA_PARAMS_TAIL;  // the copy has them
    p = &own;
  }
};
int layout_of(const RpaParams* p) { return p->layout & ~RPA_PARAMS_TAIL; }

// Workspace that a call brings.  Where a plan needs more than the one that stood in its place before, the plan is chosen by
// this: a call that ran without a workspace still does.
size_t workspace_of(const RpaParams* p) { return p->workspace ? p->workspace_bytes : 0; }

// elements of a row of queries, keys, values and outputs
int q_dim_of(const RpaParams* p) { return p->q_head_dim > 0 ? p->q_head_dim : p->head_dim; }

int esize_of(int kv_dtype) { return kv_dtype == RPA_KV_FP8_E4M3 ? 1 : 2; }

rpa::KvAddr kv_addr(const RpaParams* p) {
  rpa::KvAddr kv;
  const int es = esize_of(p->kv_dtype);
  const int64_t D = p->head_dim, H = p->num_kv_heads, P = p->page_size;
  kv.k_base = static_cast<const char*>(p->kv_cache);
  if (layout_of(p) == RPA_LAYOUT_FUSED) {
    kv.v_base = kv.k_base + D * es;
    kv.head_stride = (int32_t)(2 * D * es);
    kv.tok_stride = (int32_t)(2 * H * D * es);
  } else {
    kv.v_base = static_cast<const char*>(p->v_pages);
    kv.head_stride = (int32_t)(D * es);
    kv.tok_stride = (int32_t)(H * D * es);
  }
  kv.page_stride = (int64_t)kv.tok_stride * P;
  return kv;
}

rpa::PageTable page_table(const RpaParams* p) {
  rpa::PageTable pt;
  pt.kv_lens = p->kv_lens;
  pt.page_indices = p->page_indices;
  pt.cu_q_lens = p->cu_q_lens;
  pt.cu_kv_lens = p->cu_kv_lens;
  pt.pages_per_seq = p->pages_per_seq;
  pt.page_size = p->page_size;
  return pt;
}

rpa::SoftmaxOpts softmax_opts(float sm_scale, float soft_cap, float mask_value, int window) {
  rpa::SoftmaxOpts s;
  s.sm_scale = sm_scale;
  s.soft_cap = soft_cap;
  s.mask_value = (mask_value == 0.0f) ? kDefaultMask : mask_value;
  s.window = window;
  s.sink = nullptr;
  s.xai_len = 0.f;
  s.mask_mode = RPA_MASK_CAUSAL;
  s.mask_rows_page_aligned = 0;
  s.custom_mask = nullptr;
  s.cu_mask_lens = nullptr;
  s.round_logits = 0;
  s.q_scale = 0.f;
  return s;
}

rpa::SoftmaxOpts softmax_opts(const RpaParams* p) {
  rpa::SoftmaxOpts s = softmax_opts(p->sm_scale, p->soft_cap, p->mask_value, p->sliding_window);
  s.sink = p->attention_sink;
  s.xai_len = p->xai_temperature_len;
  s.mask_mode = p->mask_mode;
  s.mask_rows_page_aligned = p->mask_rows_page_aligned;
  s.custom_mask = p->custom_mask;
  s.cu_mask_lens = p->cu_mask_lens;
  s.round_logits = p->softmax_dtype == RPA_SOFTMAX_BF16 ? 1 : (p->softmax_dtype == RPA_SOFTMAX_F16 ? 2 : 0);
  s.q_scale = p->q_scale;
  return s;
}

int64_t kv_len_bound(int max_kv_len, int pages_per_seq, int page_size, int total_pages, bool ragged) {
  if (max_kv_len > 0) return max_kv_len;
  if (!ragged && pages_per_seq > 0) return (int64_t)pages_per_seq * page_size;
  return (int64_t)total_pages * page_size;
}

// Split-KV plan.  A split is one wave job per (row, kv head); `units` such jobs exist
// per split index and `work` is their total length in tokens.  The decode kernels hold
// `capacity` waves at once (8 per CU); measured on MI355X, one full round of equally long
// jobs beats both fewer, longer jobs (idle CUs) and many short ones (per-job prologue,
// partial write and a longer combine), so the chunk is sized to fill one round.
struct SplitPlan {
  int chunk;
  int splits;
};

int wave_capacity() { return rpa::compute_units() * 8; }

// one_round: the slots are all there is (one workgroup per CU), and a piece too many costs a round of its own.
SplitPlan plan_splits(int64_t max_len, int window, int64_t units, int64_t work, int forced, int min_chunk,
                      int capacity, bool one_round = false) {
  int64_t eff = max_len;
  if (window > 0 && eff > (int64_t)window + 31) eff = (int64_t)window + 31;
  if (eff < 1) eff = 1;
  if (units < 1) units = 1;
  const bool uniform = (work <= 0 || work >= units * eff);  // every row as long as the bound (or unknown)
  if (uniform) work = units * eff;
  int64_t chunk;
  if (forced > 0) {
    chunk = (eff + forced - 1) / forced;
  } else {
    // Every row wastes about half a job on its remainder.  With ragged rows the jobs differ
    // in length and the dispatcher does not fill CUs evenly, so a plan that uses every slot
    // spills into a second, nearly empty round: aim at 85 % of the slots (measured optimum
    // on the mixed Llama-3-8B batch: 82-88 %).
    const int64_t room = (uniform ? (int64_t)capacity : (int64_t)capacity * 17 / 20) - units / 2;
    chunk = room > 0 ? (work + room - 1) / room : eff;
    if (chunk < min_chunk) chunk = min_chunk;
    if (chunk > eff) chunk = eff;
    // equal-length rows: spread the remainder over all splits instead of one short job
    if (uniform) chunk = (eff + (eff + chunk - 1) / chunk - 1) / ((eff + chunk - 1) / chunk);
  }
  chunk = (chunk + 31) / 32 * 32;
  if (chunk < 32) chunk = 32;
  // (37 rows of 1024 tokens: 7 pieces of 160 are 259 workgroups, 56 us; 6 of 192 are 222, 43 us)
  if (one_round && forced <= 0 && uniform && units <= capacity)
    while ((eff + chunk - 1) / chunk * units > capacity) chunk += 32;
  int64_t splits = (eff + chunk - 1) / chunk;
  if (splits < 1) splits = 1;
  SplitPlan sp;
  sp.chunk = (int)chunk;
  sp.splits = (int)splits;
  return sp;
}

int decode_wave_capacity(const RpaParams* p);

SplitPlan decode_plan(const RpaParams* p) {
  const int64_t bound = kv_len_bound(p->max_kv_len, p->pages_per_seq, p->page_size, p->total_pages,
                                     p->cu_kv_lens != nullptr);
  const int G = p->num_q_heads / p->num_kv_heads;
  const int64_t per_row = (int64_t)p->num_kv_heads * ((G + 15) / 16);
  const int64_t units = (int64_t)p->decode_end * per_row;
  int64_t work = p->sum_decode_kv_len > 0 ? p->sum_decode_kv_len * per_row : 0;
  if (p->sliding_window > 0) work = 0;  // visible lengths are not the raw lengths
  SplitPlan sp = plan_splits(bound, p->sliding_window, units, work, p->num_splits,
                             rpa::tuning().decode_min_chunk, decode_wave_capacity(p));
  // Short pieces of small batches: 128 or 256 tokens where that gives all pieces, counted by the longest row, a wave slot at
  // once, at two waves per CU for bf16 (a workgroup that finds its row ended still takes its turn at the dispatcher), or
  // where a row's partials outgrow the merge.  4 rows of 1000..4095 tokens x 8 heads 22.8 us at 64, 16.9 at 128, 14.6 at
  // 256; e4m3 8 rows of 500..2047 17.8 / 13.1 / 13.8; one row of 16000 x 1 head 21.3 -> 15.1.  From about 160 tokens on
  // the pieces fill the chip and longer ones lose; bf16 on pages that are
  // no multiple of 16, whose tokens cost more, gains by the merge only.
  if (p->num_splits > 0 || sp.splits <= 1 || sp.chunk > 128) return sp;
  int64_t eff = std::max<int64_t>(bound, 1);
  if (p->sliding_window > 0) eff = std::min(eff, (int64_t)p->sliding_window + 31);
  const bool fp8 = p->kv_dtype == RPA_KV_FP8_E4M3, small_pages = p->page_size % 16 != 0;
  const int64_t slots = decode_wave_capacity(p), most = fp8 || small_pages ? slots : slots / 2;
  auto splits = [&](int chunk) { return (eff + chunk - 1) / chunk; };
  auto crowded = [&](int chunk) {
    return splits(chunk) * units > slots * 3 / 4 && (fp8 ? chunk < 128 : !small_pages);
  };
  int chunk = 64;
  while (chunk < sp.chunk) chunk *= 2;
  while (chunk < 256 && (splits(chunk) > 64 || crowded(chunk))) chunk *= 2;
  if (chunk > sp.chunk && splits(chunk) * units <= most && (!small_pages || fp8 || splits(sp.chunk) > 64)) {
    sp.chunk = chunk;
    sp.splits = (int)splits(chunk);
  }
  return sp;
}

// Balanced decode plan: a fixed number of waves (every wave slot of the GPU once) share the
// 32-token blocks of the batch evenly; the device works the partition out from kv_lens.
bool decode_balanced() { return rpa::tuning().decode_balanced != 0; }

// The balanced plan pays for itself on ragged batches.  Rows of one known length (the host's
// sum equals rows x bound) split evenly under the fixed plan already, and small batches the
// fixed plan does not split at all finish in one launch with no partial rows.
int decode_waves_per_wg(const RpaParams* p);
int decode_wgs(const RpaParams* p);
int64_t decode_kv_bytes(const RpaParams* p);
size_t balanced_bytes(const RpaParams* p);

// Whether the fixed plan's pieces come out even enough.  Its launch starts streaming about 4 us earlier than the balanced
// one (no prefix sum, no piece to look up), but what its pieces leave uneven is lost: with one piece per slot at best
// (72 MB), on rows of nearly one length (mean at least 0.7 of the longest), or cut finely (24 pieces), the start wins.
// 128 rows of 256..512 tokens x 2 heads 25.0 -> 19.0 us, 16 x 1024 x 8 heads 23.9 -> 18.5, 16 x 2048..16384 x 2 heads
// 39.2 -> 35.3; beyond: 16 x 512..4096 x 8 heads 40.2 balanced against 47.8.
bool fixed_is_even(const RpaParams* p, const SplitPlan& fixed) {
  const int64_t bytes = decode_kv_bytes(p);
  if (bytes <= (72ll << 20)) return true;
  // many short rows, none of them cut: the dispatcher evens them out, and nothing is left to merge (250 rows of 100..200
  // tokens x 8 heads 42.5 -> 32.3 us, 500 x 200..400 x 2 heads 43.8 -> 32.7; rows of up to 600 tokens about level)
  if (fixed.splits <= 1 && (int64_t)p->max_kv_len * 2 * p->head_dim * esize_of(p->kv_dtype) <= (256ll << 10) && p->max_kv_len > 0)
    return true;
  if (p->sliding_window > 0 || p->sum_decode_kv_len <= 0 || p->max_kv_len <= 0) return false;
  if (fixed.splits >= 24 && bytes <= (256ll << 20)) return true;
  return bytes <= (128ll << 20) && p->sum_decode_kv_len * 10 >= (int64_t)p->decode_end * p->max_kv_len * 7;
}

bool use_balanced(const RpaParams* p, const SplitPlan& fixed) {
  if (!decode_balanced()) return false;
  if (p->num_splits == 1) return false;  // the caller asked for whole rows: one launch, no merge pass
  // Rows the fixed plan leaves whole finish in one launch with no merge pass: right for small,
  // latency-bound batches.  A large ragged batch is still better dealt out evenly -- one job per
  // (row, kv head) of very different lengths, about one per wave slot, ends with the longest row
  // (128 rows of 128..4096 tokens: 228 -> 205 us, 200 rows of 1000..3000: 351 -> 295 us).
  if (fixed.splits <= 1 && decode_kv_bytes(p) < (64ll << 20)) return false;
  if (p->num_splits > 0) return true;
  if (fixed_is_even(p, fixed)) return false;
  // too little work to hand every workgroup its minimum piece: latency-bound, keep the launch count low
  const int64_t bound = kv_len_bound(p->max_kv_len, p->pages_per_seq, p->page_size, p->total_pages,
                                     p->cu_kv_lens != nullptr);
  const int nw = decode_waves_per_wg(p);
  const int64_t units = (int64_t)((p->num_kv_heads + nw - 1) / nw) * ((p->num_q_heads / p->num_kv_heads + 15) / 16);
  const int64_t min_blocks = std::max(1, rpa::tuning().decode_min_chunk / 32);
  if ((int64_t)p->decode_end * ((bound + 31) / 32) * units <= (int64_t)decode_wgs(p) * min_blocks)
    return false;
  const bool equal_lengths = p->sum_decode_kv_len > 0 && p->max_kv_len > 0 &&
                             p->sum_decode_kv_len == (int64_t)p->decode_end * p->max_kv_len;
  // a sliding window clips every longer row to the same length: once the mean length reaches
  // the window most rows are clipped and the batch is as good as uniform
  if (equal_lengths || (p->sliding_window > 0 && p->sum_decode_kv_len >= (int64_t)p->decode_end * p->sliding_window)) {
    // even pieces, unless most of a last round of them is empty: 67 rows behind a window of 4096 x 8 kv heads are 1072 pieces
    // on 1024 slots, two rounds for the work of one (e4m3 138.0 -> 93.1 us, bf16 261 -> 172; 140 rows of 1024 tokens 137 -> 104;
    // at 0.78 of the rounds the two plans are level).  Whole rows need no merge: 150 x 512 tokens e4m3 (167 MB) 41.6 against 43.3
    // us, bf16 (333 MB) 76.0 against 67.1.  On pages that are no multiple of 16 the balanced plan has a cache write in front, which it pays
    // for many times over (pages of 16, tokens brought along: the 67 rows 311 -> 211 us, e4m3 243 -> 137; 140 x 1024 tokens
    // 160 -> 122, 36 x 4096 163 -> 119, 130 x 2048 x 4 heads 160 -> 111).  Without the room that the balanced plan needs the
    // rows stay on the fixed one, which needs less, or nothing.
    if (fixed.splits <= 1 && decode_kv_bytes(p) < (256ll << 20)) return false;
    if (workspace_of(p) < balanced_bytes(p)) return false;
    const int64_t waves = (int64_t)p->decode_end * p->num_kv_heads * ((p->num_q_heads / p->num_kv_heads + 15) / 16) * fixed.splits;
    const int64_t slots = decode_wave_capacity(p), rounds = (waves + slots - 1) / slots;
    return waves * 10 < rounds * slots * 7;
  }
  return true;
}

// The pieces of rpa_decode_row_kernel, a workgroup of eight waves for each (row, kv head, piece), one to a CU; splits == 0: it does
// not take the rows.
//   * Rows of up to 128 KiB per kv head (255 bf16 tokens, twice that in e4m3, or a short window), as many as there are CUs: whole, in
//     one launch.  10.2 -> 7.5 us for a few rows (the second launch is the host's time too), 64 rows of 64..255 x 4 heads
//     15.7 -> 12.1; a few rows of 511 tokens: 7.8 against 9.6, a CU draws about 40 bytes per ns from beyond its L1.
//   * Even rows whose pieces are one round of the CUs, nearly all of them, where those of single waves are more than a workgroup per
//     CU: a piece of 224 bf16 tokens and more is a
//     stream of eight waves that start together and are merged in LDS, against single waves on 64 to 256 tokens or on a share of the
//     balanced plan, each with a start and a partial row of its own.  32 rows of 800..1000 tokens x 8 heads 31.5 -> 24.1 us, 8 of
//     800..1000 (4 pieces) 14.0 -> 12.0, 2 of 8000 (16 pieces) 21.5 -> 17.9, e4m3 32 x 1600..2000 34.7 -> 26.6.  Not below that
//     (8 x 500 in 4 pieces 9.1 -> 9.8; e4m3, whose blocks cost more, 16 x 1000 in 2 13.5 -> 14.3), nor beyond 640 KiB (whole rows 1 MiB) a piece, where every plan streams at the memory's rate
//     (16 x 8000 e4m3 46.8 -> 49.2), nor for uneven rows (mean under 0.75 of the longest, 0.85 in more than two
//     pieces: 16 x 500..2000 x 8 heads, 0.78 and 2 pieces, 26.3 -> 24.8, x 2 heads, 8 pieces, 12.2 -> 13.6)
//     or a quarter of the CUs idle (48 rows x 2 heads x 800..1000 16.5 -> 18.0), unless the rows are whole and of up to 512 KiB
//     (24 x 800..1000 x 8 heads 25.2 -> 23.2).
//   Most of these borders stand on one or two shapes.  194 drawn decode batches (1 to 400 rows of 20 to 32000 tokens, head counts, page
//   sizes and options at random) and 78 buckets, against the kernels and plans that took them before there were pieces by workgroups:
//   0.86 of the time in the geometric mean, none slower by more than 0.5 %.
SplitPlan row_plan(const RpaParams* p, const SplitPlan& fixed) {
  const SplitPlan none = {0, 0};
  const rpa::Tuning& tune = rpa::tuning();
  if (p->num_splits > 0 || tune.decode_row_kb == 0) return none;
  int64_t longest = std::max<int64_t>(1, kv_len_bound(p->max_kv_len, p->pages_per_seq, p->page_size, p->total_pages, p->cu_kv_lens != nullptr));
  if (p->sliding_window > 0) longest = std::min(longest, (int64_t)p->sliding_window + 31);
  const int64_t token = 2 * (q_dim_of(p) == 64 && p->kv_dtype == RPA_KV_BF16 ? 64 : p->head_dim) * esize_of(p->kv_dtype);
  const int64_t units = (int64_t)p->decode_end * p->num_kv_heads * ((p->num_q_heads / p->num_kv_heads + 15) / 16);
  const int64_t cus = rpa::compute_units(), kb = tune.decode_row_kb >= 0 ? tune.decode_row_kb : 128;
  auto pieces = [&](int64_t n) {
    SplitPlan sp;
    sp.chunk = (int)(((longest + n - 1) / n + 31) / 32 * 32);
    sp.splits = (int)((longest + sp.chunk - 1) / sp.chunk);
    return sp;
  };
  if (tune.decode_row_pieces > 0) return pieces(tune.decode_row_pieces);
  if (units > cus || units < 1) return none;
  if (longest * token <= (kb << 10)) return fixed.splits > 1 ? pieces(1) : none;
  const SplitPlan sp = pieces(cus / units);
  const bool even = p->sum_decode_kv_len > 0 && p->max_kv_len > 0 &&
                    (p->sliding_window > 0 && p->max_kv_len > p->sliding_window
                         ? p->sum_decode_kv_len >= (int64_t)p->decode_end * p->sliding_window
                         : p->sum_decode_kv_len * 20 >= (int64_t)p->decode_end * p->max_kv_len * (sp.splits <= 2 ? 15 : 17));
  if (!even || fixed.splits * units <= 2 * cus) return none;
  const bool fp8 = p->kv_dtype == RPA_KV_FP8_E4M3;
  const int64_t bytes = sp.chunk * token, least = (fp8 ? 160 : 112) << 10, most = sp.splits > 1 ? 640 << 10 : 1 << 20;
  const int64_t busy = cus / units * units;
  if (busy * 8 < cus * 7 && !(busy * 4 >= cus * 3 && sp.splits == 1 && bytes <= (512 << 10))) return none;
  // (a call that brings less workspace than this needs stays on the plan that stood here before)
  const size_t need = sp.splits > 1 ? (size_t)p->decode_end * sp.splits * p->num_q_heads * (p->head_dim + 2) * sizeof(float) : 0;
  return bytes >= least && bytes <= most && need <= workspace_of(p) ? sp : none;
}

struct DecodeChoice {
  bool balanced, rows;  // neither: pieces of single waves
  SplitPlan sp;         // (not balanced)
};
DecodeChoice decode_choice(const RpaParams* p, bool token_rows = false) {
  DecodeChoice c = {false, false, decode_plan(p)};
  const SplitPlan r = row_plan(p, c.sp);
  if (r.splits > 0) {
    c.rows = true;
    c.sp = r;
    return c;
  }
  c.balanced = !token_rows && use_balanced(p, c.sp);
  return c;
}

// Bytes of KV the decode rows will read, as far as the host knows (its sum of lengths, or rows
// times the length bound).
int64_t decode_kv_bytes(const RpaParams* p) {
  int64_t tokens = p->sum_decode_kv_len;
  if (tokens <= 0)
    tokens = (int64_t)p->decode_end * kv_len_bound(p->max_kv_len, p->pages_per_seq, p->page_size, p->total_pages,
                                                   p->cu_kv_lens != nullptr);
  if (p->sliding_window > 0) tokens = std::min(tokens, (int64_t)p->decode_end * (p->sliding_window + 31));
  return tokens * 2 * p->num_kv_heads * (q_dim_of(p) == 64 && p->kv_dtype == RPA_KV_BF16 ? 64 : p->head_dim) * esize_of(p->kv_dtype);
}

// The decode rows' row of the shape table (rpa_shapes.h): waves of a workgroup = neighbouring kv heads walked
// together (their rows are adjacent in the cache), and the waves resident at once = bytes in flight.
const rpa::ShapeRule& decode_shape(const RpaParams* p) {
  rpa::ShapeKey k = {};
  k.stage = rpa::kStageDecode;
  k.kv_bits = 8 * esize_of(p->kv_dtype);
  k.head_dim = p->head_dim;
  k.heads = p->num_q_heads / p->num_kv_heads;
  k.kv_bytes = decode_kv_bytes(p);
  return rpa::select_shape(k);
}

int decode_waves_per_wg(const RpaParams* p) {
  const int forced = rpa::tuning().decode_waves_per_wg;
  const int nw = forced > 0 ? forced : decode_shape(p).waves_per_wg;
  return std::max(1, std::min(std::min(nw, 4), p->num_kv_heads));
}

// Always a whole number of workgroups, and never a workgroup count between one and two per CU, which the
// dispatcher spreads unevenly (1152 waves in 4-wave workgroups: 133 us on C2).
int decode_wave_capacity(const RpaParams* p) {
  const int env = rpa::tuning().decode_wave_capacity;
  if (env > 0) return env;
  const int cus = rpa::compute_units();
  const int nw = decode_waves_per_wg(p);
  return std::max(nw, cus * decode_shape(p).resident_x8 / 8 / nw * nw);
}

// Waves of a workgroup of the fixed plan: two up to 256 MB (its pieces spread over more CUs), else the shape table's.
int decode_fixed_waves(const RpaParams* p) {
  const int nw = decode_waves_per_wg(p);
  return rpa::tuning().decode_waves_per_wg > 0 || decode_kv_bytes(p) >= (256ll << 20) ? nw : std::min(nw, 2);
}

int decode_wgs(const RpaParams* p) { return std::max(1, decode_wave_capacity(p) / decode_waves_per_wg(p)); }

int check_hip(hipError_t e, const char* what) {
  if (e == hipSuccess) return RPA_OK;
  return fail(RPA_EHIP, "%s: %s", what, hipGetErrorString(e));
}

size_t rows256_bytes(const RpaParams* p, const SplitPlan& sp) {
  return (size_t)p->decode_end * sp.splits * p->num_q_heads * (p->head_dim + 2) * sizeof(float);
}

// head_dim 256, decode rows: split like the fixed plan when there are too few rows to fill the GPU.
// Pieces of 256 tokens and more, for every wave slot at two waves per SIMD, except
//   * 64 or 128 tokens while those are at most 512 pieces: such a batch is a chain of blocks and nothing else (one row of
//     700 tokens x 8 heads, bf16, with the prefetch 34.9 -> 13.4 us, 8 rows of 300..3000 x 2 heads 35.6 -> 18.9; 20000 tokens x 8 heads, 1250
//     pieces of 128: 40.7 -> 51.7, the merge);
//   * twice the slots where the rows alone take more than half of them and differ in length: a piece was longer than most
//     rows there, and the long rows were waited for (180 rows of 500..3000 tokens x 8 heads 277 -> 238 us);
// both only while their partial rows stay below 16 MiB (a few long rows among many short ones take a slot per piece of
// the longest), far inside the array of rpa_attention_noalloc, and fit the workspace that the call brings.
SplitPlan rows256_plan(const RpaParams* p) {
  const int64_t bound = kv_len_bound(p->max_kv_len, p->pages_per_seq, p->page_size, p->total_pages,
                                     p->cu_kv_lens != nullptr);
  const int G = p->num_q_heads / p->num_kv_heads;
  const int64_t per_row = (int64_t)p->num_kv_heads * ((G + 15) / 16);
  const int64_t units = (int64_t)p->decode_end * per_row;
  int64_t work = p->sum_decode_kv_len > 0 ? p->sum_decode_kv_len * per_row : 0;
  if (p->sliding_window > 0) work = 0;
  const int slots = wave_capacity();
  const int64_t seen = p->sliding_window > 0 ? std::min<int64_t>(bound, (int64_t)p->sliding_window + 31) : bound;
  const int64_t tokens = work > 0 ? std::min(work, units * seen) : units * seen;
  const int min_chunk = tokens <= 64 * (slots / 4) ? 64 : tokens <= 128 * (slots / 4) ? 128 : 256;
  const bool ragged = work > 0 && work < units * seen && units * 2 > slots;
  if (min_chunk < 256 || ragged) {
    const SplitPlan sp = plan_splits(bound, p->sliding_window, units, work, p->num_splits, min_chunk, ragged ? 2 * slots : slots);
    const size_t need = sp.splits > 1 ? rows256_bytes(p, sp) : 0;
    if (need <= ((size_t)16 << 20) && need <= workspace_of(p)) return sp;
  }
  return plan_splits(bound, p->sliding_window, units, work, p->num_splits, 256, slots);
}

size_t rows256_workspace(const RpaParams* p) {
  if (p->decode_end <= 0) return 0;
  const SplitPlan sp = rows256_plan(p);
  return sp.splits <= 1 ? 0 : rows256_bytes(p, sp);
}

// head_dim 256: every query token of sequences [seq_begin, seq_end) is a row of the row kernel
// (keys / values: of decode rows whose tokens the kernel is to write)
int rows256(const RpaParams* p, int seq_begin, int seq_end, void* stream, int dist_role = 0, const void* keys = nullptr,
            const void* values = nullptr) {
  if (seq_end <= seq_begin) return RPA_OK;
  rpa::DecodeArgs a = {};
  a.q = static_cast<const uint16_t*>(p->q);
  a.out = static_cast<uint16_t*>(p->out);
  a.kv = kv_addr(p);
  a.pt = page_table(p);
  a.sm = softmax_opts(p);
  a.k_scale = p->k_scale;
  a.v_scale = p->v_scale;
  a.num_rows = seq_end;
  a.Hq = p->num_q_heads;
  a.Hkv = p->num_kv_heads;
  a.G = p->num_q_heads / p->num_kv_heads;
  a.q_dim = q_dim_of(p);
  a.fp8 = p->kv_dtype == RPA_KV_FP8_E4M3;
  a.dist = dist_role ? p->distribution : nullptr;
  a.new_k = static_cast<const char*>(keys);
  a.new_v = static_cast<const char*>(values);
  // decode rows are one token each; other sequences are bounded by the tokens of the call
  const int rows = (dist_role != 2 && seq_end <= p->decode_end) ? (seq_end - seq_begin) : p->num_tokens;
  if (seq_begin == 0 && seq_end == p->decode_end && p->mask_mode != RPA_MASK_CUSTOM) {
    const SplitPlan sp = rows256_plan(p);
    if (sp.splits > 1) {
      const size_t need = rows256_workspace(p);
      if (!p->workspace || p->workspace_bytes < need)
        return fail(RPA_EINVAL_WORKSPACE, "workspace of %zu bytes needed, %zu given", need, p->workspace_bytes);
      a.chunk = sp.chunk;
      a.max_splits = sp.splits;
      a.ws_o = static_cast<float*>(p->workspace);
      a.ws_ml = a.ws_o + (size_t)p->decode_end * sp.splits * p->num_q_heads * p->head_dim;
    }
  }
  return check_hip(rpa::launch_rows256(a, seq_begin, seq_end, rows, dist_role, static_cast<hipStream_t>(stream)),
                   "rpa rows256");
}

}  // namespace

constexpr int kTokenRows = 64;                  // query tokens
constexpr int64_t kTokenRowBytes = 64ll << 20;  // what they read, every token its whole row

// ---- rpa_attention_noalloc: the split-KV workspace as a static device array ----
// Every GPU the library is loaded on holds one copy of the array until the process ends.
constexpr size_t kNoAllocScratchBytes = (size_t)40 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];
constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

// The array's address on the current device (its name is only a host-side handle): looked up once
// per device with that device current, then kept.
int noalloc_scratch(void** out) {
  int dev = -1;
  if (int rc = check_hip(hipGetDevice(&dev), "hipGetDevice")) return rc;
  if (dev < 0 || dev >= kMaxDevices) return fail(RPA_EUNSUPPORTED, "device ordinal %d: at most %d devices", dev, kMaxDevices);
  void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!ptr) {
    if (int rc = check_hip(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)")) return rc;
    if (!ptr) return fail(RPA_EHIP, "hipGetSymbolAddress(scratch) returned a null address");
    g_scratch_ptr[dev].store(ptr, std::memory_order_release);
  }
  *out = ptr;
  return RPA_OK;
}

extern "C" {

int rpa_version(void) { return RPA_VERSION; }

const char* rpa_last_error(void) { return g_err; }

int rpa_validate(const RpaParams* given) {
  const OwnParams in(given);
  const RpaParams* p = in.p;
  if (!p) return fail(RPA_EINVAL_NULL, "params is NULL");
  if (p->num_tokens < 0 || p->num_seqs < 0 || p->num_q_heads <= 0 || p->num_kv_heads <= 0 ||
      p->head_dim <= 0 || p->page_size <= 0 || p->total_pages <= 0)
    return fail(RPA_EINVAL_SHAPE, "expected positive shape: T=%d S=%d Hq=%d Hkv=%d D=%d P=%d pages=%d",
                p->num_tokens, p->num_seqs, p->num_q_heads, p->num_kv_heads, p->head_dim,
                p->page_size, p->total_pages);
  if (p->num_q_heads % p->num_kv_heads != 0)
    return fail(RPA_EINVAL_HEADS, "expected num_q_heads=%d to be divisible by num_kv_heads=%d",
                p->num_q_heads, p->num_kv_heads);
  if (p->q_head_dim != 0 && (p->q_head_dim < 0 || p->q_head_dim > p->head_dim || p->head_dim - p->q_head_dim >= 128 ||
                             p->q_head_dim * esize_of(p->kv_dtype) % 16 != 0 || p->q_head_dim % 8 != 0))
    return fail(RPA_EUNSUPPORTED, "q_head_dim=%d: multiples of 8 (e4m3: 16) that round up to head_dim=%d", p->q_head_dim, p->head_dim);
  if (p->head_dim != 128 && p->head_dim != 256)
    return fail(RPA_EUNSUPPORTED, "head_dim=%d: 128 and 256 are built", p->head_dim);
  if (p->kv_dtype != RPA_KV_BF16 && p->kv_dtype != RPA_KV_FP8_E4M3)
    return fail(RPA_EINVAL_DTYPE, "kv_dtype=%d is not a floating point cache dtype", p->kv_dtype);
  if (layout_of(p) != RPA_LAYOUT_FUSED && layout_of(p) != RPA_LAYOUT_SPLIT)
    return fail(RPA_EINVAL_SHAPE, "layout=%d unknown", p->layout);
  if (layout_of(p) == RPA_LAYOUT_SPLIT && !p->v_pages)
    return fail(RPA_EINVAL_NULL, "split layout needs v_pages");
  if (p->sliding_window < 0) return fail(RPA_EINVAL_WINDOW, "sliding_window=%d must be positive", p->sliding_window);
  if (std::isnan(p->soft_cap)) return fail(RPA_EINVAL_SOFTCAP, "soft_cap must not be NaN");
  if (!p->distribution && (p->decode_end < 0 || p->decode_end > p->num_seqs))
    return fail(RPA_EINVAL_DISTRIBUTION, "distribution must satisfy 0 <= decode_end=%d <= num_seqs=%d",
                p->decode_end, p->num_seqs);
  if (p->num_seqs > 0) {
    if (!p->q || !p->out || !p->kv_cache || !p->kv_lens || !p->page_indices || !p->cu_q_lens)
      return fail(RPA_EINVAL_NULL, "q/out/kv_cache/kv_lens/page_indices/cu_q_lens must be non-NULL");
    if (!p->cu_kv_lens && p->pages_per_seq <= 0)
      return fail(RPA_EINVAL_SHAPE, "padded page table needs pages_per_seq > 0");
  }
  if (p->mask_value > 0.0f) return fail(RPA_EINVAL_SHAPE, "mask_value=%g must be negative", p->mask_value);
  if (p->mask_mode < RPA_MASK_CAUSAL || p->mask_mode > RPA_MASK_NONE)
    return fail(RPA_EINVAL_SHAPE, "mask_mode=%d is not an RpaMaskMode", p->mask_mode);
  if (p->mask_mode == RPA_MASK_CUSTOM && (!p->custom_mask || (!p->cu_mask_lens && !mask_as_bits(p))))
    return fail(RPA_EINVAL_NULL, "RPA_MASK_CUSTOM needs custom_mask and, where the mask is not turned into bits, cu_mask_lens");
  if (p->mask_mode == RPA_MASK_CUSTOM && p->mask_rows_page_aligned && !p->cu_kv_lens)
    return fail(RPA_EINVAL_NULL, "page-aligned mask rows need cu_kv_lens");
  if (p->softmax_dtype != RPA_SOFTMAX_F32 && p->softmax_dtype != RPA_SOFTMAX_BF16 && p->softmax_dtype != RPA_SOFTMAX_F16)
    return fail(RPA_EINVAL_DTYPE, "softmax_dtype=%d is not an RpaSoftmaxDtype", p->softmax_dtype);
  if (p->q_scale < 0.0f || std::isnan(p->q_scale))
    return fail(RPA_EINVAL_SHAPE, "q_scale=%g must be positive (0 = off)", p->q_scale);
  if (p->xai_temperature_len < 0.0f || std::isnan(p->xai_temperature_len))
    return fail(RPA_EINVAL_SHAPE, "xai_temperature_len=%g must be positive", p->xai_temperature_len);
  return RPA_OK;
}

int rpa_validate_host(const RpaParams* given, const int32_t* kv_lens, const int32_t* page_indices,
                      int64_t num_page_indices, const int32_t* cu_q_lens, const int32_t* cu_kv_lens,
                      const int32_t* distribution) {
  const OwnParams in(given);
  const RpaParams* p = in.p;
  int rc = rpa_validate(p);
  if (rc != RPA_OK) return rc;
  if (!kv_lens || !page_indices || !cu_q_lens) return fail(RPA_EINVAL_NULL, "host metadata is NULL");
  int i = 0, j = 0, k = p->num_seqs;
  if (distribution) {
    i = distribution[0]; j = distribution[1]; k = distribution[2];
    if (!(i <= j && j <= k)) return fail(RPA_EINVAL_DISTRIBUTION, "distribution must satisfy i <= j <= k, got %d, %d, %d", i, j, k);
    if (k != p->num_seqs || i != p->decode_end)
      return fail(RPA_EINVAL_DISTRIBUTION, "distribution (%d,%d,%d) disagrees with decode_end=%d num_seqs=%d", i, j, k, p->decode_end, p->num_seqs);
  } else {
    i = p->decode_end;
  }
  if (cu_q_lens[k] > p->num_tokens)
    return fail(RPA_EINVAL_SHAPE, "cu_q_lens[%d]=%d exceeds max_num_tokens=%d", k, cu_q_lens[k], p->num_tokens);
  const int P = p->page_size;
  for (int s = 0; s < k; ++s) {
    const int q_len = cu_q_lens[s + 1] - cu_q_lens[s];
    const int kv_len = kv_lens[s];
    if (q_len <= 0) return fail(RPA_EINVAL_QLEN_GT_KVLEN, "Sequence %d: q_len=%d must be > 0", s, q_len);
    if (q_len > kv_len) return fail(RPA_EINVAL_QLEN_GT_KVLEN, "Sequence %d: q_len=%d > kv_len=%d", s, q_len, kv_len);
    if (s < i && q_len != 1) return fail(RPA_EINVAL_DISTRIBUTION, "Sequence %d is in the decode range but q_len=%d", s, q_len);
    const int page_cnt = (kv_len + P - 1) / P;
    int64_t start;
    if (cu_kv_lens) {
      if (cu_kv_lens[s] % P != 0) return fail(RPA_EINVAL_SHAPE, "cu_kv_lens[%d]=%d is not page aligned", s, cu_kv_lens[s]);
      if (cu_kv_lens[s + 1] - cu_kv_lens[s] < page_cnt * P)
        return fail(RPA_EINVAL_PAGE_RANGE, "Sequence %d: page_cnt=%d does not fit cu_kv_lens", s, page_cnt);
      start = cu_kv_lens[s] / P;
    } else {
      if (page_cnt > p->pages_per_seq)
        return fail(RPA_EINVAL_PAGE_RANGE, "Sequence %d: page_cnt=%d > pages_per_seq=%d", s, page_cnt, p->pages_per_seq);
      start = (int64_t)s * p->pages_per_seq;
    }
    if (start + page_cnt > num_page_indices)
      return fail(RPA_EINVAL_PAGE_RANGE, "Sequence %d: page list [%lld, %lld) exceeds page_indices length %lld", s,
                  (long long)start, (long long)(start + page_cnt), (long long)num_page_indices);
    for (int pg = 0; pg < page_cnt; ++pg) {
      const int idx = page_indices[start + pg];
      if (idx < 0 || idx >= p->total_pages)
        return fail(RPA_EINVAL_PAGE_RANGE, "Sequence %d, page %d: index=%d out of [0, %d)", s, pg, idx, p->total_pages);
    }
    if (p->max_kv_len > 0 && kv_len > p->max_kv_len)
      return fail(RPA_EINVAL_SHAPE, "Sequence %d: kv_len=%d exceeds max_kv_len=%d", s, kv_len, p->max_kv_len);
    if (s >= i && p->max_q_len > 0 && q_len > p->max_q_len)
      return fail(RPA_EINVAL_SHAPE, "Sequence %d: q_len=%d exceeds max_q_len=%d", s, q_len, p->max_q_len);
  }
  return RPA_OK;
}

// Static-shape mode: every sequence may be a decode row, nothing is known about their lengths
// beyond the page-table bound.
static RpaParams planning_view(const RpaParams* p) {
  RpaParams q = *p;
  if (p->distribution) {
    q.decode_end = p->num_seqs;
    q.sum_decode_kv_len = 0;
  }
  return q;
}

namespace {
// Workspace of the balanced decode plan: partial rows, their (max, sum) pairs, the prefix sum of
// the rows' blocks, and one 8-byte arrival word per (row, unit, wave of the workgroup).
struct BalancedLayout {
  size_t ml, cu_blocks, counters, total;  // byte offsets
};
BalancedLayout balanced_layout(const RpaParams* p) {
  const size_t groups = (size_t)decode_wgs(p) * decode_waves_per_wg(p) * 2 * 16;
  const int nw = decode_waves_per_wg(p);
  const size_t units = (size_t)((p->num_kv_heads + nw - 1) / nw) * ((p->num_q_heads / p->num_kv_heads + 15) / 16);
  BalancedLayout l;
  l.ml = groups * p->head_dim * sizeof(float);
  l.cu_blocks = l.ml + groups * 2 * sizeof(float);
  l.counters = (l.cu_blocks + ((size_t)p->decode_end + 1) * sizeof(int32_t) + 7) & ~(size_t)7;
  l.total = l.counters + (size_t)p->decode_end * units * nw * sizeof(unsigned long long);
  return l;
}
size_t balanced_bytes(const RpaParams* p) { return balanced_layout(p).total; }
std::atomic<unsigned long long> g_decode_generation{1};

// The call with `bytes` of workspace: what it then takes is asked before there is a buffer.
RpaParams with_room(const RpaParams* p, size_t bytes) {
  static char room[1];
  RpaParams q = *p;
  q.workspace = room;  // (never read)
  q.workspace_bytes = bytes;
  return q;
}
}  // namespace

static size_t prefill_optional_workspace(const RpaParams* p);
static bool takes_token_rows(const RpaParams* p);
static size_t token_row_workspace(const RpaParams* p);

// What the decode partition cannot run without.
static size_t required_workspace_bytes(const RpaParams* p_in) {
  if (!p_in) return 0;
  const RpaParams pv = planning_view(p_in);
  const RpaParams* p = &pv;
  if (p->decode_end <= 0) return 0;
  if (p->head_dim == 256) return rows256_workspace(p);
  const DecodeChoice c = decode_choice(p);
  if (c.balanced) return balanced_layout(p).total;
  return c.sp.splits <= 1 ? 0 : (size_t)p->decode_end * c.sp.splits * p->num_q_heads * (p->head_dim + 2) * sizeof(float);
}

size_t rpa_workspace_bytes(const RpaParams* given) {
  const OwnParams in(given);
  if (!in.p) return 0;
  const RpaParams roomy = with_room(in.p, SIZE_MAX);
  const RpaParams* p = &roomy;
  const size_t need = std::max(required_workspace_bytes(p), prefill_optional_workspace(p));
  return takes_token_rows(p) ? std::max(need, token_row_workspace(p)) : need;
}

int rpa_gather_pages(const RpaParams* given, int32_t seq, void* k_out, void* v_out, int32_t max_tokens,
                     void* stream) {
  const OwnParams in(given);
  const RpaParams* p = in.p;
  int rc = rpa_validate(p);
  if (rc != RPA_OK) return rc;
  if (seq < 0 || seq >= p->num_seqs) return fail(RPA_EINVAL_SHAPE, "seq=%d out of [0, %d)", seq, p->num_seqs);
  if (!k_out || !v_out) return fail(RPA_EINVAL_NULL, "k_out/v_out is NULL");
  rpa::GatherArgs a;
  a.kv = kv_addr(p);
  a.pt = page_table(p);
  a.seq = seq;
  a.Hkv = p->num_kv_heads;
  a.head_bytes = p->head_dim * esize_of(p->kv_dtype);
  a.row_bytes = a.Hkv * a.head_bytes;
  a.k_out = k_out;
  a.v_out = v_out;
  a.max_tokens = max_tokens;
  return check_hip(rpa::launch_gather(a, static_cast<hipStream_t>(stream)), "rpa_gather_pages");
}

// The row kernels' view of a call whose query tokens are all rows of their own.
static RpaParams token_row_view(const RpaParams* p) {
  RpaParams q = *p;
  q.decode_end = p->num_tokens;
  q.sum_decode_kv_len = 0;
  q.num_splits = 0;
  return q;
}

// Whether a call that may hold chunks runs with a row per query token on the decode kernels: a few tokens on short
// contexts, where what counts is launches (cache write, decode rows, their merge, chunks, their merge: 5 x 3 us of host
// time against 2) and not that a chunk's prefix is read once per token.  (RPA_PREFILL_SPLITS asks for the prefill kernels.)
// Not a bucket of no sequences: the row kernels ask for the first one's lengths before they know how many there are.
static bool takes_token_rows(const RpaParams* p) {
  if (p->num_seqs <= 0 || p->head_dim != 128 || p->mask_mode != RPA_MASK_CAUSAL || p->num_splits > 0 || p->num_tokens <= 0 ||
      p->num_tokens > kTokenRows || rpa::tuning().prefill_splits >= 0 || (!p->distribution && p->num_seqs <= p->decode_end))
    return false;
  const RpaParams v = token_row_view(p);
  return decode_kv_bytes(&v) <= kTokenRowBytes;
}
static size_t token_row_workspace(const RpaParams* p) {
  const RpaParams v = token_row_view(p);
  const SplitPlan sp = decode_choice(&v, true).sp;
  return sp.splits <= 1 ? 0 : (size_t)v.decode_end * sp.splits * v.num_q_heads * (v.head_dim + 2) * sizeof(float);
}

// Decode rows; with keys / values the rows' own tokens are not in the cache yet and are written by these kernels.
// token_rows: every query token of the call is a row (takes_token_rows).
static int decode_rows(const RpaParams* p_in, const void* keys, const void* values, bool token_rows, void* stream) {
  const RpaParams pv = token_rows ? token_row_view(p_in) : planning_view(p_in);
  const RpaParams* p = &pv;
  if (p->decode_end <= 0) return RPA_OK;
  if (p->mask_mode == RPA_MASK_CUSTOM) return RPA_OK;  // masked rows all go through the prefill kernel
  if (p->head_dim == 256) return rows256(p, 0, p->decode_end, stream, p->distribution ? 1 : 0, keys, values);
  const DecodeChoice choice = decode_choice(p, token_rows);
  const SplitPlan& sp = choice.sp;
  rpa::DecodeArgs a;
  a.new_k = static_cast<const char*>(keys);
  a.new_v = static_cast<const char*>(values);
  a.token_rows = token_rows ? 1 : 0;
  a.num_seqs = p->num_seqs;
  a.q = static_cast<const uint16_t*>(p->q);
  a.out = static_cast<uint16_t*>(p->out);
  a.kv = kv_addr(p);
  a.pt = page_table(p);
  a.sm = softmax_opts(p);
  a.k_scale = p->k_scale;
  a.v_scale = p->v_scale;
  a.num_rows = p->decode_end;
  a.Hq = p->num_q_heads;
  a.Hkv = p->num_kv_heads;
  a.G = p->num_q_heads / p->num_kv_heads;
  a.q_dim = q_dim_of(p);
  a.chunk = sp.chunk;
  a.max_splits = sp.splits;
  a.fp8 = p->kv_dtype == RPA_KV_FP8_E4M3;
  a.ws_o = nullptr;
  a.ws_ml = nullptr;
  a.cu_blocks = nullptr;
  a.merge_counters = nullptr;
  a.generation = 0;
  a.dist = p->distribution;
  a.balanced = choice.balanced ? 1 : 0;
  a.num_wgs = decode_wgs(p);
  a.group_rows = choice.rows ? 1 : 0;
  a.waves_per_wg = a.balanced ? decode_waves_per_wg(p) : decode_fixed_waves(p);
  a.min_blocks_per_wave = std::max(1, rpa::tuning().decode_min_chunk / 32);
  a.forced_blocks_per_wave = 0;
  if (p->num_splits > 0) {  // the caller pins the partition: about num_splits pieces for the longest row
    const int64_t bound = kv_len_bound(p->max_kv_len, p->pages_per_seq, p->page_size, p->total_pages,
                                       p->cu_kv_lens != nullptr);
    a.forced_blocks_per_wave = (int32_t)std::max<int64_t>(1, ((bound + 31) / 32 + p->num_splits - 1) / p->num_splits);
  }
  if (a.balanced) {
    const size_t need = required_workspace_bytes(p);
    if (!p->workspace || p->workspace_bytes < need)
      return fail(RPA_EINVAL_WORKSPACE, "workspace of %zu bytes needed, %zu given", need, p->workspace_bytes);
    const BalancedLayout lay = balanced_layout(p);
    char* ws = static_cast<char*>(p->workspace);
    a.ws_o = reinterpret_cast<float*>(ws);
    a.ws_ml = reinterpret_cast<float*>(ws + lay.ml);
    a.cu_blocks = reinterpret_cast<int32_t*>(ws + lay.cu_blocks);
    // Opt-in: the wave that arrives last at a cut row merges it, and the second launch goes.
    // Every workgroup of the balanced grid is resident from the start and ends with its cut
    // piece, so all merges fall at the very end of the kernel, where they cost what the second
    // launch costs, and the written-through partial rows cost more: it measures slower.
    if (rpa::tuning().decode_merge_in_kernel != 0 && (reinterpret_cast<uintptr_t>(ws) & 7) == 0) {
      a.merge_counters = reinterpret_cast<unsigned long long*>(ws + lay.counters);
      // 48 bits, never zero: the arrival words are never cleared, and a word of zeros must not
      // look like this call's
      a.generation = (g_decode_generation.fetch_add(1, std::memory_order_relaxed) % ((1ull << 48) - 1)) + 1;
    }
  } else if (sp.splits > 1) {
    const size_t need = token_rows ? token_row_workspace(p_in) : required_workspace_bytes(p);
    if (!p->workspace || p->workspace_bytes < need)
      return fail(RPA_EINVAL_WORKSPACE, "workspace of %zu bytes needed, %zu given", need, p->workspace_bytes);
    a.ws_o = static_cast<float*>(p->workspace);
    a.ws_ml = a.ws_o + (size_t)p->decode_end * sp.splits * p->num_q_heads * p->head_dim;
  }
  return check_hip(rpa::launch_decode(a, static_cast<hipStream_t>(stream)), "rpa_decode");
}

int rpa_decode(const RpaParams* given, void* stream) {
  const OwnParams in(given);
  const RpaParams* p = in.p;
  const int rc = rpa_validate(p);
  if (rc != RPA_OK) return rc;
  const WorkspaceTurn turn(p->workspace);
  return decode_rows(p, nullptr, nullptr, false, stream);
}

static rpa::KvWriteArgs kv_write_args(const RpaParams* p, const void* keys, const void* values) {
  rpa::KvWriteArgs a = {};
  a.kv = kv_addr(p);
  a.pt = page_table(p);
  a.keys = static_cast<const char*>(keys);
  a.values = static_cast<const char*>(values);
  a.num_seqs = p->num_seqs;
  a.dist = p->distribution;
  a.Hkv = p->num_kv_heads;
  a.head_bytes = p->head_dim * esize_of(p->kv_dtype);
  a.src_head_bytes = q_dim_of(p) * esize_of(p->kv_dtype);
  a.num_tokens = p->num_tokens;
  return a;
}

// Whether a call's chunks are prompts whose keys and values, every token of them, the caller brings along: the kernels
// then read those rows and not the cache, and write the cache beside the attention.  (1003 tokens x 8 heads on 16-token
// pages 32.2 -> 24.3 us, on pages of 64, which the assembly kernel takes, 27.0 -> 22.1.)
static bool takes_fresh_prompts(const RpaParams* p) {
  return p->prompts_only && !p->distribution && p->decode_end == 0 && p->mask_mode != RPA_MASK_CUSTOM && q_dim_of(p) == p->head_dim &&
         p->num_seqs > 0 && p->num_tokens > 0 && !(p->head_dim == 256 && rpa::tuning().prefill_rows256 != 0) &&
         (int64_t)p->num_tokens * p->num_kv_heads * p->head_dim * esize_of(p->kv_dtype) < (int64_t(1) << 31);
}

// Whether the launch of small chunks behind prefixes (rpa_prefill_packed_kernel) may take the new tokens from the caller's rows and write them into
// the cache beside the attention.  Not with decode rows in the call, whose launch in front writes the chunks' tokens too.  A call that says
// nothing of a prefix may be all new, an address per lane and row: up to 512 tokens.
// On pages of 16 tokens and whole tiles a tile with new tokens takes twice as long as one of cached rows (an address per lane in place of one per tile), which
// outweighs the 3 us of the launch in front once the workgroups of a CU go through some of them: tokens x query heads x longest chunk in bytes of an element,
// 12 M of them being three such tiles per wave.  The call, in front -> beside, with that number: bf16 1056 tokens x 8 / 2 heads 19.1 -> 15.8 us (10 M), 1361 of up
// to 1470 on pages of 48 30.6 -> 26.3, but 1672 x 8 / 1 40.5 -> 43.3 (23 M), 1951 x 8 / 1 35.0 -> 38.6 (37 M), 1628 x 8 / 2 36.5 -> 43.2 (36 M); e4m3 1170 x 8 / 4
// 20.7 -> 18.5 (8 M), 2354 x 8 / 1 37.4 -> 39.3 (28 M).
static bool chunks_bring_tokens(const RpaParams* p, const void* keys, const void* values) {
  const int64_t longest = p->max_q_len > 0 ? p->max_q_len : p->num_tokens;
  return !p->distribution && (p->decode_end == 0 || p->mask_mode == RPA_MASK_CUSTOM) && p->head_dim == 128 && q_dim_of(p) == p->head_dim &&
         (p->max_kv_len > p->max_q_len || p->num_tokens <= 512) && ((reinterpret_cast<uintptr_t>(keys) | reinterpret_cast<uintptr_t>(values)) & 15) == 0 &&
         ((p->page_size % 32 != 0 && p->page_size != 16) || longest * p->num_tokens * p->num_q_heads * esize_of(p->kv_dtype) <= 12'000'000) &&
         (int64_t)p->num_tokens * p->num_kv_heads * p->head_dim * esize_of(p->kv_dtype) < (int64_t(1) << 31);
}

// The prefill kernels' view of a call; false when the call has no chunk for them.
// fresh: a prompt's keys / values, which the kernels read in place of the cache (takes_fresh_prompts).
static bool prefill_args(const RpaParams* p, rpa::PrefillArgs& a, const void* keys = nullptr, const void* values = nullptr) {
  const bool dyn = p->distribution != nullptr;
  if (!dyn && p->num_seqs <= p->decode_end && p->mask_mode != RPA_MASK_CUSTOM) return false;
  if (dyn && p->num_seqs <= 0) return false;
  a.head_dim = p->head_dim;
  a.q = static_cast<const uint16_t*>(p->q);
  a.out = static_cast<uint16_t*>(p->out);
  a.kv = kv_addr(p);
  a.pt = page_table(p);
  a.sm = softmax_opts(p);
  a.k_scale = p->k_scale;
  a.v_scale = p->v_scale;
  a.seq_begin = (p->mask_mode == RPA_MASK_CUSTOM || dyn) ? 0 : p->decode_end;  // dyn: the kernels read it
  a.seq_end = p->num_seqs;
  a.dist = p->distribution;
  a.Hq = p->num_q_heads;
  a.Hkv = p->num_kv_heads;
  a.G = p->num_q_heads / p->num_kv_heads;
  a.q_dim = q_dim_of(p);
  a.max_q_len = p->max_q_len > 0 ? p->max_q_len : p->num_tokens;
  a.max_kv_len = p->max_kv_len > 0 ? p->max_kv_len : 0;
  a.fp8 = p->kv_dtype == RPA_KV_FP8_E4M3;
  a.kv_splits = 1;
  a.num_tokens = p->num_tokens;
  a.ws_o = nullptr;
  a.ws_ml = nullptr;
  a.mask_bits = nullptr;
  a.mask_pitch = 0;
  a.rows_are_new = 0;
  a.page_options = rpa::page_options(p->page_size, a.kv.page_stride, 64);
  a.write_blocks = a.write_tokens = 0;
  a.write = {};
  a.tail_is_new = a.mask_words = a.saves_launch = 0;
  auto write_beside = [&]() {
    a.write = kv_write_args(p, keys, values);
    // two tokens per wave on a small launch, where the attention's own workgroups leave CUs idle
    a.write_tokens = p->num_tokens <= 2048 ? 8 : 32;
    a.write_blocks = (p->num_tokens + a.write_tokens - 1) / a.write_tokens;
  };
  if (takes_fresh_prompts(p)) {
    write_beside();
    a.rows_are_new = 1;
    a.kv.k_base = static_cast<const char*>(keys);
    a.kv.v_base = static_cast<const char*>(values);
    a.kv.head_stride = p->head_dim * esize_of(p->kv_dtype);
    a.kv.tok_stride = p->num_kv_heads * a.kv.head_stride;
    a.kv.page_stride = 0;  // (the id of the one page, whatever the table holds, adds nothing)
    a.pt.page_size = 1 << 30;  // (a.page_options stay the cache's)
  }
  // (not where the caller pins the partition: such a call agrees bit for bit with one whose composition is on the device)
  // (the mask rows of a workgroup in its LDS: two query heads per kv head and more; RPA_MASK_BITS=0 keeps a load per score, on the same kernel)
  a.mask_words = p->mask_mode == RPA_MASK_CUSTOM && !dyn && a.G >= 2 && p->max_kv_len <= (1 << 24) && p->page_size <= (1 << 24) && p->soft_cap == 0.f &&
                 a.sm.round_logits == 0 && a.sm.xai_len <= 0.f && a.sm.q_scale <= 0.f;
  // (of the call's shape alone, whether or not it brings tokens: the workspace is asked for before that is known)
  a.saves_launch = !a.rows_are_new && chunks_bring_tokens(p, keys, values);
  a.packed = p->num_splits == 0 ? rpa::prefill_packed_pieces(a) : 0;
  if (!a.packed || rpa::tuning().mask_bits == 0) a.mask_words = 0;
  if (a.packed && keys && !a.rows_are_new && chunks_bring_tokens(p, keys, values)) {
    write_beside();
    // A workgroup has a CU to itself here: those that write, which stand behind the attention's of every piece, are as few as those leave CUs for in their
    // last round, or one more is waited for (144 tokens on up to 1859, 16 / 8 heads, e4m3, 240 workgroups in three pieces: of 8 tokens each 26.4 us, of 32
    // 18.8; in front 21.7).  Where they leave none, eight tokens each (121 on up to 4098, 256 workgroups: 22.5, of 64 tokens 26.3).
    const int per = 32 / a.G, cus = rpa::compute_units();
    const int64_t wgs = (int64_t)(a.seq_end - a.seq_begin) * ((a.max_q_len + per - 1) / per) * a.Hkv * a.packed;
    for (int tokens = 8; tokens <= 64; tokens *= 2) {
      const int blocks = (p->num_tokens + tokens - 1) / tokens;
      if (wgs % cus + (int64_t)blocks * a.packed > cus) continue;
      a.write_tokens = tokens;
      a.write_blocks = blocks;
      break;
    }
    a.tail_is_new = 1;
  }
  return true;
}

// What a prefill launch can use of the workspace, none of it required: the partial rows of K/V ranges cut into
// pieces (launches that would leave most of the GPU idle), and a custom mask turned into bits by a pre-pass
// (needs a bound on the lengths; RPA_MASK_BITS=0 keeps the kernels on the caller's i32 words).
namespace {
struct PrefillWorkspace {
  int splits;
  int pitch;  // 64-bit words per bit row
  size_t split_bytes, bits_offset, bits_bytes, total;
};
PrefillWorkspace prefill_workspace(const RpaParams* p, const rpa::PrefillArgs& a) {
  PrefillWorkspace w = {};
  w.splits = rpa::prefill_kv_splits(a);
  w.split_bytes = rpa::prefill_split_workspace_bytes(a, w.splits);
  w.bits_offset = (w.split_bytes + 255) & ~(size_t)255;
  w.bits_bytes = mask_bits_bytes(p);
  w.pitch = w.bits_bytes ? (p->max_kv_len + 63) / 64 : 0;
  w.total = w.bits_bytes ? w.bits_offset + w.bits_bytes : w.split_bytes;
  return w;
}
}  // namespace

// Workspace that lets a prefill launch which would leave most of the GPU idle cut its K/V ranges into
// pieces; never required: without it the launch runs whole ranges.
static size_t prefill_optional_workspace(const RpaParams* p) {
  rpa::PrefillArgs a;
  if (!prefill_args(p, a)) return 0;
  if (p->head_dim == 256 && rpa::tuning().prefill_rows256 != 0) return 0;  // the row kernel has its own plan
  return prefill_workspace(p, a).total;
}

static int write_new_tokens(const RpaParams* p, const void* keys, const void* values, bool skip_decode_rows, void* stream);

static int prefill_launch(const RpaParams* p, rpa::PrefillArgs& a, const void* keys, const void* values, void* stream);

// keys / values: new tokens that the launch itself puts into the cache (prompts without a prefix, custom masks).
static int prefill_run(const RpaParams* p, const void* keys, const void* values, void* stream) {
  const int rc = rpa_validate(p);
  if (rc != RPA_OK) return rc;
  rpa::PrefillArgs a;
  return prefill_args(p, a, keys, values) ? prefill_launch(p, a, keys, values, stream) : RPA_OK;
}

static int prefill_launch(const RpaParams* p, rpa::PrefillArgs& a, const void* keys, const void* values, void* stream) {
  int rc;
  // 256-wide heads take the flash kernel (two 128-dim halves per row, one workgroup per CU; e4m3
  // caches staged through registers); RPA_PREFILL_ROWS256=1 sends them through the row kernel
  if (p->head_dim == 256 && rpa::tuning().prefill_rows256 != 0)
    return rows256(p, (p->mask_mode == RPA_MASK_CUSTOM || p->distribution) ? 0 : p->decode_end, p->num_seqs, stream,
                   p->distribution ? 2 : 0);
  if (p->workspace && (reinterpret_cast<uintptr_t>(p->workspace) & 15) == 0) {
    // the decode partition is done with the workspace by the time these kernels run (same stream)
    const PrefillWorkspace w = prefill_workspace(p, a);
    char* ws = static_cast<char*>(p->workspace);
    size_t bits_at = 0;
    bool cut = false, bits = false;
    if (w.bits_bytes && p->workspace_bytes >= w.total) {
      bits = true;
      bits_at = w.bits_offset;
      cut = w.splits > 1;
    } else if (w.bits_bytes && p->workspace_bytes >= w.bits_bytes) {
      bits = true;  // room for the bits alone: they save more than the pieces
    } else if (w.splits > 1 && p->workspace_bytes >= w.split_bytes) {
      cut = true;
    }
    if (cut) {
      a.kv_splits = w.splits;
      a.ws_o = reinterpret_cast<float*>(ws);
      a.ws_ml = a.ws_o + (size_t)p->num_tokens * p->num_q_heads * w.splits * p->head_dim;
    }
    if (bits) {
      a.mask_bits = reinterpret_cast<uint64_t*>(ws + bits_at);
      a.mask_pitch = w.pitch;
    }
  }
  if (a.mask_words) a.mask_bits = nullptr;
  if (keys && p->mask_mode == RPA_MASK_CUSTOM && !a.tail_is_new) {  // by the launch that makes the bits, if there is one
    if (a.mask_bits) a.write = kv_write_args(p, keys, values);
    else if ((rc = write_new_tokens(p, keys, values, false, stream)) != RPA_OK) return rc;
  }
  if (p->mask_mode == RPA_MASK_CUSTOM && !p->cu_mask_lens && !a.mask_bits && !a.mask_words)
    return fail(RPA_EINVAL_WORKSPACE, "a mask without cu_mask_lens needs rpa_workspace_bytes() of workspace");
  return check_hip(rpa::launch_prefill(a, static_cast<hipStream_t>(stream)), "rpa_prefill");
}

int rpa_upload_words(int32_t* dst, const int32_t* src, int32_t n, void* stream) {
  if (n <= 0) return RPA_OK;
  if (!dst || !src) return fail(RPA_EINVAL_NULL, "dst/src is NULL");
  return check_hip(rpa::launch_upload(dst, src, n, static_cast<hipStream_t>(stream)), "rpa_upload_words");
}

// The new tokens are in the cache already.
static int prefill_cached(const RpaParams* p, void* stream) {
  if (!p || !p->prompts_only) return prefill_run(p, nullptr, nullptr, stream);
  RpaParams q = *p;
  q.prompts_only = 0;
  return prefill_run(&q, nullptr, nullptr, stream);
}

int rpa_prefill(const RpaParams* given, void* stream) {
  const OwnParams in(given);
  const WorkspaceTurn turn(in.p ? in.p->workspace : nullptr);
  return prefill_cached(in.p, stream);
}

int rpa_mask_needs_starts(const RpaParams* given) {
  const OwnParams in(given);
  return in.p && in.p->mask_mode == RPA_MASK_CUSTOM && !mask_as_bits(in.p) ? 1 : 0;
}

// (narrow heads: only the kernels that know of the zeros behind 64 dims)
static bool rows_take_new_tokens(const RpaParams* p) {
  const int d = q_dim_of(p);
  return d == p->head_dim || (d == 64 && p->kv_dtype == RPA_KV_BF16 && rpa::tuning().decode_merge_in_kernel == 0);
}

// Whether the decode kernels take their rows' new tokens from the caller's keys / values and write them into the cache
// (not the balanced plan on pages that are no multiple of 16 tokens).  256-wide rows: up to 768 MB of cache, where a launch in front is a
// part of the call that one notices (5 rows of 1396..8992 e4m3 tokens x 2 heads 22.2 -> 17.6 us, one of 700 bf16 x 8 heads 11.9 -> 9.7,
// 32 of 300..3000 x 4 heads 50.6 -> 47.6, 64 of 300..3000 e4m3 x 8 heads, 0.4 GB, 95.6 -> 89.4, 180 of 500..3000, 0.6 GB, 244 -> 239); the
// same on bf16, 1.3 GB, 447 -> 447.5.
static bool decode_takes_new_tokens(const RpaParams* p_in) {
  if (p_in->head_dim == 256) {
    const RpaParams p = planning_view(p_in);
    return p_in->mask_mode != RPA_MASK_CUSTOM && decode_kv_bytes(&p) <= (768ll << 20);
  }
  if (p_in->head_dim != 128 || p_in->mask_mode == RPA_MASK_CUSTOM || !rows_take_new_tokens(p_in)) return false;
  if (p_in->page_size % 16 == 0) return true;
  const RpaParams p = planning_view(p_in);
  return !decode_choice(&p).balanced;
}

static int write_new_tokens(const RpaParams* p, const void* keys, const void* values, bool skip_decode_rows, void* stream) {
  rpa::KvWriteArgs a = kv_write_args(p, keys, values);
  a.skip_decode_rows = skip_decode_rows ? 1 : 0;
  a.seq_begin = skip_decode_rows && !p->distribution ? p->decode_end : 0;
  return check_hip(rpa::launch_kv_write(a, static_cast<hipStream_t>(stream)), "rpa_kv_write");
}

// Whether the decode rows of a call write their tokens themselves.  (With chunks behind the rows their tokens need a launch
// anyway, and it takes the rows' along: 317.1 -> 316.7 us, 47.3 -> 47.1, 162.7 -> 162.3 for mixed batches.  With the
// composition on the device there are chunks in few calls, and the launch for them ends at once: 30 rows of 100..700 tokens
// in a bucket of 32 24.4 -> 22.6 us.)
static bool decode_rows_write(const RpaParams* p) {
  const bool chunks = !p->distribution && p->num_seqs > p->decode_end;
  return !chunks && decode_takes_new_tokens(p);
}

int rpa_attention_update(const RpaParams* given, const void* keys, const void* values, void* stream) {
  const OwnParams in(given);
  const RpaParams* p = in.p;
  int rc = rpa_validate(p);
  if (rc != RPA_OK) return rc;
  if (!keys != !values) return fail(RPA_EINVAL_NULL, "keys and values must be given together");
  const WorkspaceTurn turn(p->workspace);
  if (takes_token_rows(p) && p->workspace_bytes >= token_row_workspace(p)) {
    const bool with_rows = keys && rows_take_new_tokens(p);
    if (keys && !with_rows && (rc = write_new_tokens(p, keys, values, false, stream)) != RPA_OK) return rc;
    return decode_rows(p, with_rows ? keys : nullptr, with_rows ? values : nullptr, true, stream);
  }
  if (keys && (takes_fresh_prompts(p) || mask_as_bits(p))) return prefill_run(p, keys, values, stream);
  // chunks alone: their plan is made once, and says who writes their tokens
  rpa::PrefillArgs a;
  const bool chunks = keys && chunks_bring_tokens(p, keys, values);
  if (chunks) {
    if (!prefill_args(p, a, keys, values)) return RPA_OK;
    if (!a.tail_is_new && (rc = write_new_tokens(p, keys, values, false, stream)) != RPA_OK) return rc;
    return prefill_launch(p, a, a.tail_is_new ? keys : nullptr, values, stream);
  }
  const bool fused = keys && decode_rows_write(p);
  if (keys && !fused && (rc = write_new_tokens(p, keys, values, false, stream)) != RPA_OK) return rc;
  if ((rc = decode_rows(p, fused ? keys : nullptr, fused ? values : nullptr, false, stream)) != RPA_OK) return rc;
  if (fused && (rc = write_new_tokens(p, keys, values, true, stream)) != RPA_OK) return rc;
  return prefill_cached(p, stream);
}

int rpa_attention(const RpaParams* p, void* stream) { return rpa_attention_update(p, nullptr, nullptr, stream); }

static bool prefill_brings_tokens(const RpaParams* p, const void* keys, const void* values) {
  rpa::PrefillArgs a;
  return chunks_bring_tokens(p, keys, values) && prefill_args(p, a, keys, values) && a.tail_is_new;
}

int rpa_describe_plan(const RpaParams* given, char* buf, size_t len) {
  const OwnParams in(given);
  const RpaParams* p_in = in.p;
  int rc = rpa_validate(p_in);
  if (rc != RPA_OK) return rc;
  if (!buf || len == 0) return fail(RPA_EINVAL_NULL, "buf is NULL or empty");
  const RpaParams roomy = with_room(p_in, SIZE_MAX);
  p_in = &roomy;
  const RpaParams pv = planning_view(p_in);
  const RpaParams* p = &pv;
  size_t at = 0;
  auto put = [&](const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    const size_t from = std::min(at, len - 1);
    const int n = vsnprintf(buf + from, len - from, fmt, ap);
    va_end(ap);
    if (n > 0) at += (size_t)n;
  };
  buf[0] = 0;
  auto put_rows = [&](const char* what, const RpaParams* v, bool token_rows, size_t workspace) {
    const rpa::ShapeRule& r = decode_shape(v);
    const DecodeChoice c = decode_choice(v, token_rows);
    const SplitPlan& sp = c.sp;
    const bool bal = c.balanced, whole = c.rows;
    put("%s: shape=%s kernel=%s rows=%d", what, r.name,
        whole ? "rpa_decode_row_kernel" : bal ? "rpa_decode_balanced_kernel" : "rpa_decode_splitkv_kernel", v->decode_end);
    if (!whole) put(" waves_per_wg=%d", bal ? decode_waves_per_wg(v) : decode_fixed_waves(v));
    if (bal) put(" resident_waves=%d merge=rpa_combine_balanced_kernel", decode_wave_capacity(v));
    else if (!whole || sp.splits > 1) put(" pieces_per_row=%d chunk=%d merge=%s", sp.splits, sp.chunk, sp.splits > 1 ? "rpa_combine_kernel" : "none");
    put(" workspace=%zu\n", workspace);
  };
  if (takes_token_rows(p_in)) {
    const RpaParams v = token_row_view(p_in);
    put_rows("whole call", &v, true, token_row_workspace(p_in));
  }
  if (p->decode_end > 0 && p->mask_mode != RPA_MASK_CUSTOM) {
    if (p->head_dim == 256)
      put("decode: shape=%s kernel=rpa_rows256_kernel rows=%d pieces_per_row=%d workspace=%zu\n", decode_shape(p).name, p->decode_end,
          rows256_plan(p).splits, required_workspace_bytes(p_in));
    else put_rows("decode", p, false, required_workspace_bytes(p_in));
  }
  rpa::PrefillArgs a;
  if (prefill_args(p_in, a)) {
    if (p->head_dim == 256 && rpa::tuning().prefill_rows256 != 0) {
      put("prefill: kernel=rpa_rows256_kernel (RPA_PREFILL_ROWS256)\n");
    } else {
      const rpa::ShapeRule& r = rpa::prefill_shape_of(a);
      const char* kernel = r.kernel == rpa::kKernelPrefillPipe     ? "rpa_prefill_pipe_kernel"
                           : r.kernel == rpa::kKernelPrefillStaged ? "rpa_prefill_staged_kernel"
                           : r.kernel == rpa::kKernelPrefillWide   ? "rpa_prefill_async_kernel_wide"
                                                                   : "rpa_prefill_async_kernel";
      const PrefillWorkspace w = prefill_workspace(p_in, a);
      // (a launch that reads the mask's words has the room for bits all the same: new tokens that are not on 16 bytes may send it elsewhere)
      put("prefill: shape=%s kernel=%s tile=%dx%dx%d kv_pieces_with_workspace=%d mask_bits=%s optional_workspace=%zu\n",
          r.name, kernel, r.tile_q, r.tile_heads, r.tile_kv, w.splits, w.bits_bytes && !a.mask_words ? "yes" : "no", w.total);
      if (rpa::prefill_by_streams(a)) put("prefill, long sequences: one after the other\n");
      if (a.packed)
        put("prefill, small launch: kernel=rpa_prefill_packed_kernel instead, columns=%d tile=%dx%dx32\n", 32, 32 / a.G, a.G);
    }
  }
  const bool rows = takes_token_rows(p_in), prompts = !rows && takes_fresh_prompts(p_in);
  const bool by_rows = rows ? rows_take_new_tokens(p_in) : !prompts && decode_rows_write(p_in);
  alignas(16) static const char some_rows[16] = {};  // (aligned ones)
  const bool beside = !rows && (prompts || prefill_brings_tokens(p_in, some_rows, some_rows));
  put("new tokens: written by %s\n", !rows && !beside && mask_as_bits(p_in) ? "the launch that makes bits of the mask"
                                     : beside                           ? "workgroups of the prefill launch, which reads the caller's rows"
                                     : !by_rows                         ? "rpa_kv_write_kernel, in front"
                                     : p_in->distribution && !rows      ? "the decode kernels, those of chunks by rpa_kv_write_kernel"
                                                                        : "the decode kernels");
  return (int)std::min<size_t>(at, 0x7fffffff);
}

size_t rpa_noalloc_max_workspace_bytes(void) { return kNoAllocScratchBytes; }

int rpa_attention_noalloc(const RpaParams* given, void* stream) {
  const OwnParams in(given);
  const RpaParams* p = in.p;
  int rc = rpa_validate(p);
  if (rc != RPA_OK) return rc;
  const RpaParams view = with_room(p, kNoAllocScratchBytes);
  const size_t need = required_workspace_bytes(&view);  // (a prefill launch cuts its K/V ranges only if the array has the room)
  if (need > kNoAllocScratchBytes)
    return fail(RPA_EINVAL_WORKSPACE,
                "this batch needs a split-KV workspace of %zu bytes, the built-in one holds %zu: call rpa_attention "
                "with a workspace of your own",
                need, kNoAllocScratchBytes);
  RpaParams q = *p;
  q.workspace = nullptr;
  q.workspace_bytes = 0;
  if (need > 0 || prefill_optional_workspace(p) > 0) {
    void* ptr = nullptr;
    if ((rc = noalloc_scratch(&ptr)) != RPA_OK) return rc;
    q.workspace = ptr;  // the device address, never the array's name
    q.workspace_bytes = kNoAllocScratchBytes;
  }
  // Nothing in the workspace has to start at zero: partial rows, their (max, sum) pairs and the block
  // prefix sums are all written by the decode kernel before the merge pass reads them.
  return rpa_attention(&q, stream);
}

int rpa_kv_write(const RpaParams* given, const void* keys, const void* values, void* stream) {
  const OwnParams in(given);
  const RpaParams* p = in.p;
  int rc = rpa_validate(p);
  if (rc != RPA_OK) return rc;
  if (!keys || !values) return fail(RPA_EINVAL_NULL, "keys/values is NULL");
  return write_new_tokens(p, keys, values, false, stream);
}

// ---------------------------------------------------------------- MLA ----

static int mla_wgs();
static float mla_logit_scale(const RpaMlaParams* p);

// The smallest piece of a row.  Partial rows are bf16, so a row that is cut is rounded once more than a whole one: batches of
// rows up to 256 tokens are left whole (their result is 2.3e-3 from the 64-bit one, in pieces of 64 it was 2.8e-3).  That is
// also the faster plan from 16 rows on (128 heads, rows of 100..255 tokens: 64 rows 36.0 -> 32.4 us, 200 rows 64.1 -> 36.5),
// but not for a few (4 rows 25.3 -> 29.1; 16 heads 16.3 -> 20.6).
constexpr int kMlaWholeRow = 256;
static int64_t mla_longest(const RpaMlaParams* p) {
  const int64_t longest = kv_len_bound(p->max_kv_len, p->pages_per_seq, p->page_size, p->total_pages, p->cu_kv_lens != nullptr);
  return std::max<int64_t>(1, p->sliding_window > 0 ? std::min(longest, (int64_t)p->sliding_window + 31) : longest);
}
static int mla_min_piece(const RpaMlaParams* p) {
  return mla_longest(p) <= kMlaWholeRow ? kMlaWholeRow : std::max(1, rpa::tuning().mla_min_chunk);
}

// What the choice of an MLA kernel depends on.
static rpa::MlaDecodeArgs mla_key_args(const RpaMlaParams* p, int64_t rows, bool token_rows) {
  rpa::MlaDecodeArgs a = {};
  a.pt.page_size = p->page_size;
  a.sm.soft_cap = p->soft_cap;
  a.sm.sm_scale = mla_logit_scale(p);
  a.sm.window = p->sliding_window;
  a.fp8 = p->cache_dtype == RPA_KV_FP8_E4M3 ? 1 : 0;
  a.Hq = p->num_q_heads;
  a.row_stride = p->row_stride;
  a.num_rows = (int32_t)rows;
  a.num_seqs = p->num_seqs;
  a.rows_are_tokens = token_rows ? 1 : 0;
  return a;
}

// How a call is cut.  wgs: pieces or shares that run at once; waves: the kernels of a wave per tile (rpa_mla_waves.hip), `siblings` workgroups of
// 16 heads per piece.
struct MlaPlan {
  SplitPlan sp;
  const rpa::ShapeRule* rule;
  int wgs, siblings, token_groups;
  bool waves, balanced;
};

// Whether a call runs on a wave per tile, with 16 heads a workgroup.  What a piece costs besides its tiles is half of the other kernels', what
// a tile costs grows with every 16 heads: so by the work, in rounds of 64 tokens x 16 heads per CU.  us, other kernels -> these, and the rounds:
//   16 heads           64 rows of 2047..16383 bf16 128 -> 113, e4m3 119 -> 76, on pages of 16 130 -> 114 and 137 -> 78; small ones on pages of 16 1.05 .. 1.4 x, on whole
//                      tiles level, e4m3 under a round 1.0 .. 0.93 x (2 of 559..1861 12.6 -> 13.6) but for whole rows (5 of 115..210 16.0 -> 12.3)
//   32 heads, e4m3     the same rows 125 -> 105 (72), 128 of 500 28.2 -> 18.5 (8); bf16 133 -> 141 (72), 30.5 -> 32.0 (9.8), 128 of 500 26.9 -> 21.4 (7.8), on
//                      pages of 16 35.3 -> 31.9 (9.8), 141 -> 145 (72); e4m3 in between 23 of 177..6038 29.3 -> 30.7 (8), 12 of 7548..9184 34.8 -> 37.1 (12), 32 of 2133..14199
//                      61.7 -> 58.9 (30); bf16 selections of 9 rows x 64 pages 22.1 -> 21.6 (4), of 23 32.5 -> 34.1 (12)
//   64 heads, bf16     20 rows of 300..1500 28.0 -> 24.5 (4.4), 54 of 300..800 31.0 -> 31.8 (7.3), on pages of 16 33.4 -> 31.7; 32 of 1000..4000 41.9 -> 45.0 (20);
//                      e4m3 5 of 2829..6230 28.6 -> 23.1 (6), 11 of 4297..4690 33.8 -> 35.1 (12), 49 of 873..1449 37.7 -> 41.8 (14), on pages of 16 17 of 399..8919
//                      47.4 -> 46.1 (21), 77 of 435..3187 66.4 -> 73.6 (36); selections of 12 rows x 64 pages 35.3 -> 33.8 (12), of 32 52.2 -> 57.2 (32), single tokens 31 of 1024
//                      28.2 -> 25.9 (8), 24 of 2048 34.7 -> 37.1 (12)
//   128 heads          one row of 4000 25.1 -> 15.8 (2), 8 of 300..1500 26.7 -> 22.8 (3.5), 20 33.1 -> 34.1 (8.8), on pages of 16 36.9 -> 34.1, e4m3 39.7 -> 33.1;
//                      54 of 300..800 37.6 -> 45.8 (14.5); selections of 4 rows x 64 pages 33.3 -> 26.3 (8), 12 of 2048 tokens 39.9 -> 39.4 (12)
// Rows that stay whole (up to 256 tokens) are short beside what a workgroup costs anyway: there by the workgroups, in rounds of the CUs.  351 drawn
// batches of rows and chunk tokens, best limit 0.75 .. 0.9 rounds for 32 heads, 0.6 .. 0.75 (pages under a tile 1.25 .. 1.75) for 64, 1.4 .. 1.7 (e4m3 2.0 .. 2.1)
// for 128: 128 heads, 78 rows of 67 tokens 20.7 -> 27.2 (2.4 rounds), 130 of 75 21.1 -> 44.3 (4.1), 32 heads 162 of 89 13.9 -> 20.1 (1.3).  So too for e4m3 rows of
// a few hundred tokens on whole tiles: 82 of 777 x 64 heads 42.8 -> 47.4 (1.3 rounds), 192 of 242 x 32 heads 33.1 -> 37.4 (1.5).
//
// 16 heads take it on pages under a tile, and on whole tiles but for e4m3 rows cut into pieces under a round (above) and bf16 selections of whole pages under 4
// rounds (bf16 rows of several lengths: see mla_plan).  Selections: the three tiles that a workgroup of the other kernel has asked for ahead are 111 KB, the
// eight of four waves arrive behind one another's waits.  200 drawn selections, inputs that change from call to call, shared tiles -> these: 9 rows of
// 4096 tokens 21.1 -> 23.5 us (2.2 rounds), 11 of 2048..2688 20.4 -> 22.4, 13 of 4096 23.9 -> 25.9 (3.2); around 4 rounds either, 16 of 4096 25.8 -> 27.3, with
// fewer pages in use 23.1 -> 22.5; 24 of 4096 32.9 -> 32.9 (6), 32 40.7 -> 37.9 (8), 64 of 8192 105 -> 92.7 (32).  Throughout: e4m3 0.75 .. 1.03 x the time,
// single tokens 0.86 .. 1.01, pages of 16 0.86 .. 1.03.
static bool mla_takes_waves(const RpaMlaParams* p, int64_t rows, bool token_rows, bool sparse) {
  const int blocks = (p->num_q_heads + 15) / 16;
  const int64_t longest = mla_longest(p);
  const int64_t tokens = p->sum_kv_len > 0 ? std::min(p->sum_kv_len, rows * longest) : rows * longest;
  const int64_t rounds = tokens * blocks / (64 * (int64_t)mla_wgs());
  const bool fp8 = p->cache_dtype == RPA_KV_FP8_E4M3, whole = p->page_size % 32 == 0;  // (pages of whole tiles: where the other kernels are at their best)
  if (blocks == 1) return !whole || (fp8 ? rounds >= 1 || longest <= kMlaWholeRow : !sparse || rounds >= 4);
  // (a chunk's tokens where their heads form no groups: 177 on 267 x 40 heads 26.7 -> 34.1, e4m3 on pages of 16 465 on 341 50.1 -> 69.9; 75 on 247 23.5 -> 15.6)
  if (token_rows && rows * blocks > 2 * (int64_t)mla_wgs()) return false;
  if (longest <= kMlaWholeRow && !sparse) {
    const int eighths = blocks > 4 ? (fp8 ? 16 : 12) : blocks > 2 ? (whole ? 6 : 10) : (fp8 ? 7 : 6);
    return 8 * rows * blocks <= (int64_t)eighths * mla_wgs();
  }
  const bool one_round = sparse || rows * blocks <= mla_wgs();
  if (blocks <= 2) {
    if (!fp8) return rounds < (sparse ? whole ? 9 : 20 : whole ? 6 : 24);
    return !whole || sparse || ((one_round || tokens >= 512 * rows) && (rounds < 5 || rounds >= 15));
  }
  if (blocks <= 4) return rounds < (fp8 ? !whole ? 22 : sparse ? 14 : one_round ? 9 : 0 : sparse ? whole ? 14 : 11 : whole ? 6 : 14);
  // (selections, one workgroup more than the CUs: 33 rows of 512 tokens 34.5 -> 42)
  return rounds < (fp8 || sparse || !whole ? 10 : 6) && (!sparse || rows * blocks <= mla_wgs());
}

// Whether a call whose query tokens could share workgroups (rpa_mla.hip, token groups) runs each of them on a wave per tile instead, its rows whole as the
// groups' are.  A group's tile costs a CU twice what four waves' tiles of one token do and its start and end (147 KB of queries, 128 KB of
// results) three times as much, but it is 8 / 4 / 2 tokens: groups win as soon as the tokens x blocks of 16 heads are some rounds of the CUs, however
// long the rows.  997 drawn calls of 16..900 new tokens on up to 8192, best limit in rounds: bf16 2.0 .. 2.25 (of 16-token pages and 16 heads 3), e4m3
// 2.75 .. 3.25, on pages under a tile, where a group's copies are slow, 2.75 .. 4.5; with the limits here 1.27 x in the geometric mean (the better
// of the two everywhere would be 1.274), none more than 4 % slower.  us, groups -> these: 16 heads, bf16, 46 tokens 29 -> 14, 163 on 512 47 -> 28, 351 on 2500 125 -> 100
// (1.4 rounds), 580 on 400 56 -> 65 (2.3); e4m3 220 on 300 47 -> 22, 735 on 2300 180 -> 141 (2.9), 1056 on 320 61 -> 84 (4.1); 32 heads e4m3 on
// pages of 16 238 on 150 54 -> 32.
static bool mla_groups_as_waves(const RpaMlaParams* p, int64_t rows) {
  const int blocks = p->num_q_heads / 16;
  const bool fp8 = p->cache_dtype == RPA_KV_FP8_E4M3, whole = p->page_size % 32 == 0;
  const int half_rounds = !fp8 ? 4 : whole ? 5 : blocks == 1 ? 8 : 6;
  return p->sliding_window <= 0 && 2 * rows * blocks <= (int64_t)half_rounds * mla_wgs();
}

static bool mla_use_balanced(const RpaMlaParams* p, const MlaPlan& plan, bool token_rows);
static MlaPlan mla_plan(const RpaMlaParams* p, int64_t rows, bool token_rows, bool sparse = false, bool waves = true) {
  const int64_t bound = kv_len_bound(p->max_kv_len, p->pages_per_seq, p->page_size, p->total_pages,
                                     p->cu_kv_lens != nullptr);
  rpa::MlaDecodeArgs a = mla_key_args(p, rows, token_rows);
  const rpa::Tuning& tune = rpa::tuning();
  MlaPlan m;
  m.rule = &rpa::select_shape(rpa::mla_shape_key(a), rpa::mla_shape_skip(a, tune));
  m.wgs = mla_wgs();
  m.waves = false;
  m.siblings = 1;
  // one workgroup per (row, split, 128 heads) and per CU; every split costs a 256 KiB
  // partial write per 128 heads, so splits are kept as few as fill the CUs once
  auto cut = [&](int64_t groups) {
    int64_t work = p->sum_kv_len > 0 ? p->sum_kv_len * groups : 0;
    if (p->sliding_window > 0) work = 0;
    // The tokens of a chunk see nearly the same, and pieces of the mean length leave a tail of the longer rows for a second round of workgroups: rows
    // that are 70 % full are cut by the longest, into what one round holds (137 tokens on 4473 x 16 heads 180 us, whole 102; 167 on 593 x 128 heads
    // 83 and 45; 34 on 3295 x 64, e4m3, 105 and 66), those of more than 3/5 of a round from 65 % on (174 on 2074 x 32, e4m3, 68 % full, 158 and 72).
    // Emptier ones stay with the mean: 88 on 3116 x 64 heads, 68 % full, 80 us and in two pieces 97, 129 on 4453 x 128, e4m3, 67 %, 208 and whole 259.
    const bool full = 20 * work >= (5 * rows * groups > 3 * m.wgs ? 13 : 14) * rows * groups * bound;
    // Of more rows than a quarter of the CUs the short ones stay whole, a merge costs more than their pieces give (101 of 259 x 128 heads 38 us, whole 29;
    // 65 of 308 x 64 27 and 18; 92 of 466 x 128 39 and 37; but e4m3 74 of 401 x 128 44, whole 54).
    const int64_t kept = p->cache_dtype == RPA_KV_FP8_E4M3 && p->num_q_heads > 64 ? 384 : 512;
    const bool keep = token_rows && 4 * rows > mla_wgs() && bound <= kept && tune.mla_min_chunk >= rpa::Tuning().mla_min_chunk;
    if (keep || (token_rows && full)) work = 0;
    const int piece = keep ? (int)kept : mla_min_piece(p);
    return plan_splits(bound, p->sliding_window, rows * groups, work, p->num_splits, piece, m.wgs, true);
  };
  m.sp = cut((p->num_q_heads + 127) / 128);
  a.max_splits = m.sp.splits;
  m.token_groups = rpa::mla_token_group_mode(a, tune, *m.rule);
  const int blocks = (p->num_q_heads + 15) / 16;
  if (m.token_groups && waves && tune.mla_waves != 0 && tune.mla_shared_tiles != 0 && (tune.mla_waves > 0 || mla_groups_as_waves(p, rows))) {
    m.token_groups = 0;
    m.waves = true;
    m.siblings = blocks;
    m.balanced = false;
    return m;
  }
  // (at most 128 heads, whatever the switch says: a share's slots in the workspace hold so many, and its line has one unit per row)
  if (waves && blocks <= 8 && tune.mla_waves != 0 && !m.token_groups && p->soft_cap == 0.f && tune.mla_shared_tiles != 0 &&
      (tune.mla_waves > 0 || mla_takes_waves(p, rows, token_rows, sparse))) {
    const MlaPlan other = m;
    m.waves = true;
    m.siblings = blocks;
    m.wgs = std::max(1, m.wgs / m.siblings);
    if (m.siblings > 1 && m.wgs > 8) m.wgs &= ~7;  // (whole eights of workgroups, see Sibling)
    m.sp = cut(1);
    // Whole long rows that are a little more than a round of workgroups, where the other kernels have pieces of them: 66 tokens on 4700 x 64 heads,
    // e4m3 on pages of 16, 170 us and 138 in three pieces, 136 of 1205 and less x 32 heads 47 and 36.
    if (token_rows && m.sp.splits <= 1 && other.sp.splits > 1 && rows * blocks > mla_wgs()) {
      m = other;
      m.balanced = false;
      return m;
    }
    // Rows of several lengths: the shortest pieces, counted by the longest row, that are one round of workgroups, if any of up to 512 tokens are.  The
    // balanced plan evens them out, but its start (prefix sums, a search) is 2 us later: 20 rows of 300..1500 x 16 heads 17.9 -> 16.1 us in pieces
    // of 128, 8 of 1000..8000 22.5 -> 20.0 of 256, 100 of 200..1000 e4m3 25.9 -> 22.7 of 512, 20 of 300..1500 x 32 heads 19.2 -> 17.4; beyond, 100 of
    // 200..1000 in pieces of 256 26.3 -> 33.4.
    const int64_t longest = mla_longest(p);
    const bool tiles16 = !sparse && !token_rows && tune.mla_waves < 0 && p->cache_dtype == RPA_KV_BF16 && p->page_size % 32 == 0;
    if (p->num_splits == 0 && !(p->sum_kv_len > 0 && p->sum_kv_len == rows * longest)) {
      bool coarse = false;
      for (int64_t chunk = mla_min_piece(p); chunk <= 512; chunk *= 2) {
        const int64_t pieces = (longest + chunk - 1) / chunk;
        if (rows * pieces > m.wgs) continue;
        // (pieces of 512 of long bf16 rows leave too many CUs idle: 31 of 137..2231 x 16 heads 20.6 -> 23.0, 7 of 5427..11524 23.2 -> 25.3, 3 of 179..14794 x 32 19.8 -> 22.3)
        if ((coarse = chunk > 256 && longest > 1024 && blocks <= 2 && tiles16)) break;
        m.sp.splits = (int)pieces;
        m.sp.chunk = (int)((longest + pieces - 1) / pieces + 31) / 32 * 32;
        m.balanced = false;
        return m;
      }
      // Longer pieces of bf16 rows on pages of whole tiles: shared tiles have less of a start than the waves' 16-token tiles and keep it up to 15 rounds
      // of 64 tokens per CU (113 drawn batches x 16 heads, shared -> waves: 12 of 5800..23203 37.4 -> 40.0, 41 of 472..7560 40.6 -> 43.6, 13.2 rounds 48.3 ->
      // 50.6; 16.3 rounds 60.3 -> 59.3, 17.2 and more 1.11 .. 1.14 x; pages of 16 1.03 .. 1.14 x, e4m3 1.11 .. 1.64 x throughout; selections: see mla_takes_waves).
      const int64_t tokens = p->sum_kv_len > 0 ? std::min(p->sum_kv_len, rows * longest) : rows * longest;
      if (coarse || (blocks == 1 && tiles16 && tokens < 15 * 64 * (int64_t)mla_wgs())) m = other;
    }
  }
  m.balanced = !sparse && mla_use_balanced(p, m, token_rows);
  return m;
}

static int mla_validate(const RpaMlaParams* p) {
  if (!p) return fail(RPA_EINVAL_NULL, "params is NULL");
  if (p->num_seqs < 0 || p->num_q_heads <= 0 || p->page_size <= 0 || p->total_pages <= 0)
    return fail(RPA_EINVAL_SHAPE, "expected positive shape");
  if (p->lkv_dim != 512 || p->rope_dim != 64)
    return fail(RPA_EUNSUPPORTED, "lkv_dim=%d rope_dim=%d: only 512+64 is built", p->lkv_dim, p->rope_dim);
  if (p->row_stride < p->rope_offset + p->rope_dim || p->rope_offset < p->lkv_dim || (p->row_stride % 8) != 0 ||
      (p->rope_offset % 8) != 0)
    return fail(RPA_EINVAL_SHAPE, "row_stride=%d rope_offset=%d do not describe [kv_c | k_pe]", p->row_stride, p->rope_offset);
  if (p->cache_dtype != RPA_KV_BF16 && p->cache_dtype != RPA_KV_FP8_E4M3)
    return fail(RPA_EINVAL_SHAPE, "cache_dtype=%d is neither RPA_KV_BF16 nor RPA_KV_FP8_E4M3", p->cache_dtype);
  if (p->cache_dtype == RPA_KV_FP8_E4M3 && ((p->row_stride % 16) != 0 || (p->rope_offset % 16) != 0))
    return fail(RPA_EINVAL_SHAPE, "fp8 latent rows: row_stride=%d and rope_offset=%d must be multiples of 16", p->row_stride,
                p->rope_offset);
  if (p->sliding_window < 0) return fail(RPA_EINVAL_WINDOW, "sliding_window=%d must be positive", p->sliding_window);
  if (p->num_seqs > 0 && (!p->ql_nope || !p->q_pe || !p->out || !p->cache_kv || !p->kv_lens || !p->page_indices || !p->cu_q_lens))
    return fail(RPA_EINVAL_NULL, "a required buffer is NULL");
  if (!p->cu_kv_lens && p->pages_per_seq <= 0 && p->num_seqs > 0)
    return fail(RPA_EINVAL_SHAPE, "padded page table needs pages_per_seq > 0");
  return RPA_OK;
}

static int mla_wgs() {
  const int forced = rpa::tuning().mla_wg_capacity;
  return std::max(1, forced > 0 ? forced : rpa::compute_units());
}

// same criteria as the MHA decode path: ragged sequence rows that need splitting
static bool mla_use_balanced(const RpaMlaParams* p, const MlaPlan& plan, bool token_rows) {
  const SplitPlan& fixed = plan.sp;
  const bool on = rpa::tuning().mla_balanced != 0;
  if (!on || token_rows || p->num_splits == 1) return false;
  if (plan.waves && mla_min_piece(p) >= kMlaWholeRow) return false;  // (rows of up to 256 tokens stay whole: see there)
  // Rows the fixed plan leaves whole: one workgroup job per row.  With many more jobs than
  // workgroup slots the dispatcher evens them out by itself; with up to two per slot the kernel
  // ends with the longest rows, and dealing the tiles out evenly pays (300 rows of 1000..8000
  // tokens: 832 -> 673 us; 256 rows of 2048..16384: 1214 -> 1013 us; 1000 rows of 200..2000:
  // 617 -> 659 us, so not there).
  if (fixed.splits <= 1 && (int64_t)p->num_seqs * ((p->num_q_heads + 127) / 128) > 2 * (int64_t)plan.wgs) return false;
  if (p->num_splits > 0) return true;
  const int64_t bound = kv_len_bound(p->max_kv_len, p->pages_per_seq, p->page_size, p->total_pages,
                                     p->cu_kv_lens != nullptr);
  const int64_t units = (p->num_q_heads + 127) / 128;
  const int64_t min_tiles = std::max(1, mla_min_piece(p) / 32);
  if ((int64_t)p->num_seqs * ((bound + 31) / 32) * units <= (int64_t)plan.wgs * min_tiles) return false;
  const bool equal_lengths = p->sum_kv_len > 0 && p->max_kv_len > 0 &&
                             p->sum_kv_len == (int64_t)p->num_seqs * p->max_kv_len;
  return !equal_lengths;
}

static size_t mla_workspace(const RpaMlaParams* p, int64_t rows, const MlaPlan& plan) {
  if (plan.balanced) return (size_t)plan.wgs * 2 * 128 * (p->lkv_dim + 2) * sizeof(float) + ((size_t)p->num_seqs + 1) * sizeof(int32_t);
  if (plan.sp.splits <= 1) return 0;
  return (size_t)rows * plan.sp.splits * p->num_q_heads * (p->lkv_dim + 2) * sizeof(float);
}

static size_t mla_workspace(const RpaMlaParams* p, int64_t rows, bool token_rows, bool sparse = false) {
  const rpa::TuningOfCall tuning;
  if (!p || p->num_seqs <= 0 || rows <= 0) return 0;
  return mla_workspace(p, rows, mla_plan(p, rows, token_rows, sparse));
}

size_t rpa_mla_workspace_bytes(const RpaMlaParams* p) { return mla_workspace(p, p ? p->num_seqs : 0, false); }

size_t rpa_mla_attention_workspace_bytes(const RpaMlaParams* p) {
  return mla_workspace(p, p ? p->num_tokens : 0, true);
}

// the scalar scales of the logits fold into sm_scale (they multiply the dot product before the soft cap)
static float mla_logit_scale(const RpaMlaParams* p) {
  return p->sm_scale * (p->k_scale > 0.f ? p->k_scale : 1.0f) * (p->q_scale > 0.f ? p->q_scale : 1.0f);
}

// new_kv_c, new_k_pe: the sequences' new tokens where the kernels are to put them into the cache (not with token_rows).
// sparse: the rows' tables and lengths, which the kernels write first.
static int mla_run(const RpaMlaParams* p, void* stream, bool token_rows, const void* new_kv_c = nullptr, const void* new_k_pe = nullptr,
                   const rpa::SparseMlaArgs* sparse = nullptr) {
  const rpa::TuningOfCall tuning;
  int rc = mla_validate(p);
  if (rc != RPA_OK) return rc;
  if (p->num_seqs <= 0) return RPA_OK;
  if (!token_rows && p->num_seqs > p->num_tokens)
    return fail(RPA_EINVAL_SHAPE, "decode rows=%d exceed tokens=%d", p->num_seqs, p->num_tokens);
  const int64_t rows = token_rows ? p->num_tokens : p->num_seqs;
  if (rows <= 0) return RPA_OK;
  MlaPlan plan = mla_plan(p, rows, token_rows, sparse != nullptr);
  // (a call that brings the room of the plan that stood here before stays on it)
  if (plan.waves && mla_workspace(p, rows, plan) > (p->workspace ? p->workspace_bytes : 0)) plan = mla_plan(p, rows, token_rows, sparse != nullptr, false);
  const SplitPlan& sp = plan.sp;
  rpa::MlaDecodeArgs a;
  a.sparse = {};
  if (sparse) a.sparse = *sparse;
  a.extra_rows = a.sparse.extra;
  a.new_kv_c = static_cast<const char*>(new_kv_c);
  a.new_k_pe = static_cast<const char*>(new_k_pe);
  a.ql_nope = static_cast<const uint16_t*>(p->ql_nope);
  a.q_pe = static_cast<const uint16_t*>(p->q_pe);
  a.out = static_cast<uint16_t*>(p->out);
  a.cache = static_cast<const char*>(p->cache_kv);
  a.pt.kv_lens = p->kv_lens;
  a.pt.page_indices = p->page_indices;
  a.pt.cu_q_lens = p->cu_q_lens;
  a.pt.cu_kv_lens = p->cu_kv_lens;
  a.pt.pages_per_seq = p->pages_per_seq;
  a.pt.page_size = p->page_size;
  a.sm = softmax_opts(mla_logit_scale(p), p->soft_cap, p->mask_value, p->sliding_window);
  a.out_scale = p->v_scale > 0.f ? p->v_scale : 1.0f;
  a.dist = p->distribution;
  a.fp8 = p->cache_dtype == RPA_KV_FP8_E4M3 ? 1 : 0;
  if (p->distribution && !token_rows)
    return fail(RPA_EUNSUPPORTED, "rpa_mla_decode takes the batch composition from the host: use rpa_mla_attention");
  a.num_rows = (int32_t)rows;
  a.num_seqs = p->num_seqs;
  a.rows_are_tokens = token_rows ? 1 : 0;
  a.Hq = p->num_q_heads;
  a.row_stride = p->row_stride;
  a.rope_offset = p->rope_offset;
  a.chunk = sp.chunk;
  a.max_splits = sp.splits;
  a.ws_o = nullptr;
  a.ws_ml = nullptr;
  a.cu_tiles = nullptr;
  a.balanced = plan.balanced ? 1 : 0;
  a.num_wgs = plan.wgs;
  a.waves = plan.waves ? 1 : 0;
  a.siblings = plan.siblings;
  a.min_tiles_per_wg = std::max(1, mla_min_piece(p) / 32);
  a.forced_tiles_per_wg = 0;
  a.piece_pad = rpa::tuning().mla_piece_pad >= 0
                    ? rpa::tuning().mla_piece_pad
                    : plan.waves
                          ? 8  // (a wave per tile: 6 .. 14 within 1 %; 3 loses 3 % on 64 rows of 2047..16383 e4m3 tokens, 10 % on short rows)
                    : rpa::mla_takes_wide_p16(a, true)
                          ? 12  // (the wide kernels' in the shape table)
                          : plan.rule->piece_pad;
  if (p->num_splits > 0) {
    const int64_t bound = kv_len_bound(p->max_kv_len, p->pages_per_seq, p->page_size, p->total_pages,
                                       p->cu_kv_lens != nullptr);
    a.forced_tiles_per_wg = (int32_t)std::max<int64_t>(1, ((bound + 31) / 32 + p->num_splits - 1) / p->num_splits);
  }
  if (a.balanced) {
    const size_t need = mla_workspace(p, rows, plan);
    if (!p->workspace || p->workspace_bytes < need)
      return fail(RPA_EINVAL_WORKSPACE, "workspace of %zu bytes needed, %zu given", need, p->workspace_bytes);
    // partial rows are bf16 (the workspace is sized for f32 rows: room to spare)
    a.ws_o = static_cast<uint16_t*>(p->workspace);
    a.ws_ml = reinterpret_cast<float*>(a.ws_o + (size_t)a.num_wgs * 2 * 128 * p->lkv_dim);
    a.cu_tiles = reinterpret_cast<int32_t*>(a.ws_ml + (size_t)a.num_wgs * 2 * 128 * 2);
  } else if (sp.splits > 1) {
    const size_t need = mla_workspace(p, rows, plan);
    if (!p->workspace || p->workspace_bytes < need)
      return fail(RPA_EINVAL_WORKSPACE, "workspace of %zu bytes needed, %zu given", need, p->workspace_bytes);
    a.ws_o = static_cast<uint16_t*>(p->workspace);
    a.ws_ml = reinterpret_cast<float*>(a.ws_o + (size_t)rows * sp.splits * p->num_q_heads * p->lkv_dim);
  }
  return check_hip(rpa::launch_mla_decode(a, static_cast<hipStream_t>(stream)),
                   token_rows ? "rpa_mla_attention" : "rpa_mla_decode");
}

int rpa_mla_describe_plan(const RpaMlaParams* p, int token_rows, char* buf, size_t len) {
  int rc = mla_validate(p);
  if (rc != RPA_OK) return rc;
  if (!buf || len == 0) return fail(RPA_EINVAL_NULL, "buf is NULL or empty");
  const int64_t rows = token_rows ? p->num_tokens : p->num_seqs;
  const MlaPlan plan = mla_plan(p, std::max<int64_t>(rows, 1), token_rows != 0);
  const rpa::ShapeRule& r = *plan.rule;
  const bool bal = rows > 0 && plan.balanced;
  static const char* const kGroups[] = {"off", "eight_waves_compiled", "eight_waves", "wide"};
  const int tg = plan.token_groups;
  const bool waves = plan.waves, p16 = !tg && !waves && rpa::mla_takes_wide_p16(mla_key_args(p, rows, token_rows != 0), true);
  return snprintf(buf, len, "mla: shape=%s rows=%lld waves_per_wg=%d heads_per_wg=%d share=%d token_groups=%s plan=%s "
                  "pieces_per_row=%d workgroups=%d workspace=%zu%s\n",
                  waves ? "mla_waves" : r.name, (long long)rows, waves || tg == 3 || p16 ? 4 : r.waves_per_wg, waves ? 16 : tg ? 128 : r.tile_heads,
                  waves || tg ? 1 : r.share, kGroups[tg], bal ? "balanced" : "fixed", bal ? 0 : plan.sp.splits, bal ? plan.wgs * plan.siblings : 0,
                  mla_workspace(p, rows, token_rows != 0), waves ? " (a wave per tile, 16 heads per workgroup)" : p16 ? " (the wide loop of pages of 16 tokens)" : "");
}

int rpa_mla_decode(const RpaMlaParams* p, void* stream) {
  const WorkspaceTurn turn(p ? p->workspace : nullptr);
  return mla_run(p, stream, false);
}

int rpa_mla_attention(const RpaMlaParams* p, void* stream) {
  const WorkspaceTurn turn(p ? p->workspace : nullptr);
  return mla_run(p, stream, true);
}

int rpa_mla_kv_write(const RpaMlaParams* p, const void* new_kv_c, const void* new_k_pe, void* stream) {
  int rc = mla_validate(p);
  if (rc != RPA_OK) return rc;
  if (!new_kv_c || !new_k_pe) return fail(RPA_EINVAL_NULL, "new_kv_c/new_k_pe is NULL");
  if (p->num_seqs <= 0 || p->num_tokens <= 0) return RPA_OK;
  rpa::MlaWriteArgs a;
  a.cache = static_cast<char*>(const_cast<void*>(p->cache_kv));
  a.pt.kv_lens = p->kv_lens;
  a.pt.page_indices = p->page_indices;
  a.pt.cu_q_lens = p->cu_q_lens;
  a.pt.cu_kv_lens = p->cu_kv_lens;
  a.pt.pages_per_seq = p->pages_per_seq;
  a.pt.page_size = p->page_size;
  a.new_kv_c = static_cast<const char*>(new_kv_c);
  a.new_k_pe = static_cast<const char*>(new_k_pe);
  a.fp8 = p->cache_dtype == RPA_KV_FP8_E4M3 ? 1 : 0;
  a.num_tokens = p->num_tokens;
  a.num_seqs = p->num_seqs;
  a.dist = p->distribution;
  a.row_stride = p->row_stride;
  a.rope_offset = p->rope_offset;
  return check_hip(rpa::launch_mla_kv_write(a, static_cast<hipStream_t>(stream)), "rpa_mla_kv_write");
}

int rpa_mla_attention_update(const RpaMlaParams* p, const void* new_kv_c, const void* new_k_pe, int token_rows,
                             void* stream) {
  const WorkspaceTurn turn(p ? p->workspace : nullptr);
  if (!new_kv_c && !new_k_pe) return mla_run(p, stream, token_rows != 0);
  if (!token_rows && new_kv_c && new_k_pe) return mla_run(p, stream, false, new_kv_c, new_k_pe);
  const int rc = rpa_mla_kv_write(p, new_kv_c, new_k_pe, stream);
  return rc != RPA_OK ? rc : mla_run(p, stream, token_rows != 0);
}

// ---- sparse attention: the dense kernels over a page table per query token ----
namespace {
// The call the dense kernels see: a decode row per query token.
RpaMlaParams sparse_view(const RpaMlaParams* p, const RpaMlaSparse* s) {
  RpaMlaParams v = *p;
  const bool rows = s->k_pages_max <= 0;
  v.num_seqs = p->num_tokens;
  v.cu_kv_lens = nullptr;
  if (rows) v.page_size = 1;
  const int entries = rows ? s->topk_count : s->k_pages_max;
  v.pages_per_seq = (entries + 31) & ~31;  // (rows of the table share no cache line)
  // a selection is as long as it can be, or as its sequence is: rows of one length, as far as the host knows (the fixed plan's
  // even pieces, 32 rows x 4096 tokens 52.5 -> 46 us against the balanced plan)
  int64_t bound = (int64_t)entries * v.page_size;
  if (s->pages_per_seq > 0) bound = std::min(bound, (int64_t)s->pages_per_seq * p->page_size);
  v.max_kv_len = (int32_t)bound;
  v.sum_kv_len = p->num_tokens * bound;
  v.num_splits = 0;
  v.distribution = nullptr;
  return v;
}

// Workspace: what the view's plan needs, then the lengths and the tables (on a cache line of its own from wherever the workspace
// begins, see rpa_dsa.h).
constexpr size_t kLine = 128;
struct SparseLayout {
  size_t kv_lens, table, extra, total;
};
SparseLayout sparse_layout(const RpaMlaParams* p, const RpaMlaSparse* s, const RpaMlaParams& view) {
  auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
  const size_t T = (size_t)p->num_tokens;
  SparseLayout l;
  l.kv_lens = up(mla_workspace(&view, view.num_seqs, false, true));
  l.table = l.kv_lens + up(T * sizeof(int32_t));
  l.extra = l.table + up(T * view.pages_per_seq * sizeof(int32_t) + kLine);
  l.total = l.extra + (s->k_pages_max > 0 ? 0 : (T + 1) * p->row_stride * (p->cache_dtype == RPA_KV_FP8_E4M3 ? 1 : 2));
  return l;
}
}  // namespace

size_t rpa_mla_sparse_workspace_bytes(const RpaMlaParams* p, const RpaMlaSparse* s) {
  if (!p || !s || p->num_tokens <= 0) return 0;
  return sparse_layout(p, s, sparse_view(p, s)).total;
}

int rpa_mla_sparse_attention(const RpaMlaParams* p, const RpaMlaSparse* s, const void* new_kv_c, const void* new_k_pe,
                             void* stream) {
  int rc = mla_validate(p);
  if (rc != RPA_OK) return rc;
  if (!s || !s->topk || !p->cu_kv_lens) return fail(RPA_EINVAL_NULL, "a selection and a ragged page table are needed");
  if (!new_kv_c != !new_k_pe) return fail(RPA_EINVAL_NULL, "new_kv_c and new_k_pe must be given together");
  if (p->num_tokens <= 0 || p->num_seqs <= 0) return RPA_OK;
  const bool rows = s->k_pages_max <= 0;
  if (s->topk_count < (s->topk_is_pages ? 0 : 1) || s->topk_stride < s->topk_count || s->num_page_indices <= 0 || (!rows && s->pages_per_seq <= 0) ||
      (rows && s->topk_is_pages))
    return fail(RPA_EINVAL_SHAPE, "selection of %d entries (stride %d), %d pages per sequence, %d page ids", s->topk_count,
                s->topk_stride, s->pages_per_seq, s->num_page_indices);
  if ((int64_t)p->total_pages * p->page_size > 0x7fffffffLL || (int64_t)s->k_pages_max * p->page_size > 0x7fffffffLL)
    return fail(RPA_EUNSUPPORTED, "%d pages of %d tokens: more than 2^31 rows", p->total_pages, p->page_size);
  RpaMlaParams v = sparse_view(p, s);
  const SparseLayout l = sparse_layout(p, s, v);
  if (!p->workspace || p->workspace_bytes < l.total || (reinterpret_cast<uintptr_t>(p->workspace) & 15) != 0)
    return fail(RPA_EINVAL_WORKSPACE, "workspace of %zu bytes needed (aligned to 16), %zu given", l.total, p->workspace_bytes);
  const WorkspaceTurn turn(p->workspace);
  char* ws = static_cast<char*>(p->workspace);
  rpa::SparseMlaArgs a = {};
  a.pt.kv_lens = p->kv_lens;
  a.pt.page_indices = p->page_indices;
  a.pt.cu_q_lens = p->cu_q_lens;
  a.pt.cu_kv_lens = p->cu_kv_lens;
  a.pt.pages_per_seq = 0;
  a.pt.page_size = p->page_size;
  a.num_page_indices = s->num_page_indices;
  a.num_tokens = p->num_tokens;
  a.num_seqs = p->num_seqs;
  a.topk = s->topk;
  a.topk_count = s->topk_count;
  a.topk_stride = s->topk_stride;
  a.topk_is_pages = s->topk_is_pages;
  a.pages_per_seq = s->pages_per_seq;
  a.k_pages_max = rows ? 0 : s->k_pages_max;
  a.total_pages = p->total_pages;
  a.cache = static_cast<char*>(const_cast<void*>(p->cache_kv));
  a.row_stride = p->row_stride;
  a.rope_offset = p->rope_offset;
  a.fp8 = p->cache_dtype == RPA_KV_FP8_E4M3 ? 1 : 0;
  a.new_kv_c = static_cast<const char*>(new_kv_c);
  a.new_k_pe = static_cast<const char*>(new_k_pe);
  a.table = reinterpret_cast<int32_t*>((reinterpret_cast<uintptr_t>(ws + l.table) + kLine - 1) & ~(uintptr_t)(kLine - 1));
  a.table_stride = v.pages_per_seq;
  a.kv_len_out = reinterpret_cast<int32_t*>(ws + l.kv_lens);
  a.extra = rows ? ws + l.extra : nullptr;
  v.kv_lens = a.kv_len_out;
  v.page_indices = a.table;
  v.workspace_bytes = l.kv_lens;
  return mla_run(&v, stream, false, nullptr, nullptr, &a);
}

}  // extern "C"
