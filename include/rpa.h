/*
 * rpa.h -- C ABI of the MI355X (gfx950) ragged paged attention library.
 *
 * The reference project (sglang-jax) has no native FFI on this path: its
 * operator boundary is a jitted Python callable.  Each entry point below names
 * the reference callable it stands in for (paths relative to the reference
 * checkout, python/sgl_jax/srt/...).  A jax.ffi custom call, a ctypes stub or
 * any other host binds exactly these symbols.
 *
 * Conventions
 *   - every pointer marked "device" is caller-owned device memory; the library
 *     never allocates or frees device memory and never synchronises a stream;
 *   - every launch is enqueued on the hipStream_t passed as `stream` (NULL is
 *     the legacy default stream), so calls are graph-capturable;
 *   - functions return RPA_OK (0) or a negative RpaStatus; rpa_last_error()
 *     returns a thread-local, human readable description of the last failure;
 *   - calls may come from several threads; the launches of two calls on one workspace do not mix, but
 *     calls that share a workspace are still ordered by the caller: on one stream, or by events;
 *   - metadata (kv_lens, page_indices, cu_q_lens, cu_kv_lens) is read on the
 *     device only.  Host copies can be checked with rpa_validate_host().
 */
#ifndef RPA_MI355_H_
#define RPA_MI355_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define RPA_VERSION 100 /* 0.1.0 */

/* The entry points below are the library's ONLY dynamic symbols: it is built with hidden default
 * visibility, so nothing else of it can collide with, or be interposed by, a host process. */
#if defined(__GNUC__) || defined(__clang__)
#define RPA_API __attribute__((visibility("default")))
#else
#define RPA_API
#endif

typedef enum RpaStatus {
  RPA_OK = 0,
  RPA_EINVAL_SHAPE = -1,
  RPA_EINVAL_DTYPE = -2,
  RPA_EINVAL_HEADS = -3,
  RPA_EINVAL_PAGE_RANGE = -4,
  RPA_EINVAL_QLEN_GT_KVLEN = -5,
  RPA_EINVAL_WINDOW = -6,
  RPA_EINVAL_SOFTCAP = -7,
  RPA_EINVAL_WORKSPACE = -8,
  RPA_EHIP = -9,
  RPA_EINVAL_DISTRIBUTION = -10,
  RPA_EUNSUPPORTED = -11,
  RPA_EINVAL_NULL = -12
} RpaStatus;

typedef enum RpaKvDtype {
  RPA_KV_BF16 = 0,
  RPA_KV_FP8_E4M3 = 1 /* OCP e4m3fn, max 448 */
} RpaKvDtype;

typedef enum RpaSoftmaxDtype {
  RPA_SOFTMAX_F32 = 0,
  RPA_SOFTMAX_BF16 = 1,
  RPA_SOFTMAX_F16 = 2
} RpaSoftmaxDtype;

typedef enum RpaMaskMode {
  RPA_MASK_CAUSAL = 0, /* query j of a sequence sees tokens <= kv_len - q_len + j */
  RPA_MASK_CUSTOM = 1, /* causal = 0 with custom_mask (speculative tree verification) */
  RPA_MASK_NONE = 2    /* causal = 0 without a mask: every query sees all kv_len tokens */
} RpaMaskMode;

typedef enum RpaLayout {
  /* one buffer [pages, P, 2*Hkv, D], heads stored K0,V0,K1,V1,...
   * (mem_cache/memory_pool.py:56-91, 580-588) */
  RPA_LAYOUT_FUSED = 0,
  /* two buffers k_pages, v_pages [pages, P, Hkv, D]
   * (kernels/ragged_paged_attention/ragged_paged_attention_v3.py:96-97) */
  RPA_LAYOUT_SPLIT = 1,
  /* added to one of the two: the caller's RpaParams has the fields behind `distribution`, q_head_dim and prompts_only.
   * Without it they are taken as 0 and not read, so that a caller compiled against a header that did not have them
   * keeps working */
  RPA_PARAMS_TAIL = 0x100
} RpaLayout;

/*
 * One ragged paged attention call.  Field meanings follow the arguments of
 * ragged_paged_attention (ragged_paged_attention_v3.py:1667-1700) and of
 * ref_ragged_paged_attention (same file, :94-114).
 */
typedef struct RpaParams {
  /* ---- device buffers ---- */
  const void* q;              /* bf16 [T, Hq, D] */
  void* out;                  /* bf16 [T, Hq, D]; rows >= cu_q_lens[num_seqs] untouched */
  const void* kv_cache;       /* FUSED: the cache; SPLIT: k_pages */
  const void* v_pages;        /* SPLIT only, else NULL */
  const int32_t* kv_lens;     /* i32[S]  (kv length INCLUDING the new q tokens) */
  const int32_t* page_indices;/* i32 flat (cu_kv_lens != NULL) or [S, pages_per_seq] */
  const int32_t* cu_q_lens;   /* i32[S+1] */
  const int32_t* cu_kv_lens;  /* i32[S+1] cumulative page-aligned kv lens; NULL => padded 2-D table */
  const float* k_scale;       /* f32[Hkv] dequantisation scale of K, or NULL (= 1) */
  const float* v_scale;       /* f32[Hkv] or NULL */
  void* workspace;            /* partial rows of cut K/V ranges; >= rpa_workspace_bytes() */
  size_t workspace_bytes;
  /* ---- static shape ---- */
  int32_t num_tokens;         /* T */
  int32_t num_seqs;           /* S = distribution[2]: sequences to process */
  int32_t num_q_heads;        /* Hq */
  int32_t num_kv_heads;       /* Hkv, Hq % Hkv == 0 */
  int32_t head_dim;           /* D of the cache's rows: 128 or 256.  Narrower heads (64, 80, 96, 192 ...) are stored
                               * zero-padded to the next multiple of 128 as in the reference (memory_pool.py:70; the
                               * reference pads the queries too, rpa_v3:1187-1241).  q, out, keys and values either
                               * come padded, or in their own width with q_head_dim (below) */
  int32_t page_size;          /* P */
  int32_t total_pages;
  int32_t pages_per_seq;      /* row stride of the padded table (cu_kv_lens == NULL) */
  int32_t layout;             /* RpaLayout, + RPA_PARAMS_TAIL where the last two fields are set */
  int32_t kv_dtype;           /* RpaKvDtype */
  /* ---- batch composition: distribution = (decode_end, prefill_end, num_seqs)
   *      (ragged_paged_attention_v3.py:82-91); sequences [0, decode_end) have
   *      q_len == 1, the rest any q_len >= 1 ---- */
  int32_t decode_end;
  /* ---- host-side bounds used only to size grids (never to index memory) ---- */
  int32_t max_kv_len;         /* upper bound of kv_lens[0:num_seqs]; 0 => pages_per_seq*P or total_pages*P */
  int32_t max_q_len;          /* upper bound of q_len over [decode_end, num_seqs); 0 => T.  A promise: rows of a
                                 longer sequence past the bound are not computed */
  int32_t num_splits;         /* decode split-KV count per sequence; 0 => automatic.  A call that fixes it also keeps its chunks
                                 off the kernel for small prefill launches, so that it agrees bit for bit with
                                 one whose composition is on the device */
  /* ---- options ---- */
  int32_t sliding_window;     /* 0 => off */
  float sm_scale;             /* the pipelined prefill kernel (bf16 cache on pages of 2^k >= 64 tokens, 128-wide
                                 heads, causal, no option) multiplies the bf16 queries by sm_scale * log2(e) and rounds them to bf16 once,
                                 where the reference scales the f32 scores (:149): element-wise inside the
                                 reference's rtol = atol = 2e-2, and at most 1.5e-2 of a row's norm on rows whose
                                 weight sits on one or two keys (1e-2 for every other path) */
  float soft_cap;             /* 0 => off */
  float mask_value;           /* 0 => default -0.7 * FLT_MAX */
  /* sum of kv_lens over the decode rows (host-side, balances the split plan); 0 => unknown */
  int64_t sum_decode_kv_len;
  /* ---- further options of ref_ragged_paged_attention (ragged_paged_attention_v3.py:103-113) ---- */
  const float* attention_sink;  /* device f32[Hq]: one extra logit per query head that enters only the
                                   softmax denominator (:185-196), or NULL */
  const int32_t* custom_mask;   /* device i32, flat: sequence i, query row j, token t at
                                   cu_mask_lens[i] + j * row_width_i + t; >= 1 keeps, < 1 masks (:154-163).
                                   Read only when mask_mode == RPA_MASK_CUSTOM */
  const int32_t* cu_mask_lens;  /* device i32[S+1]: cumulative q_len_i * row_width_i (:123-129, 1801-1806); may be NULL
                                   where rpa_mask_needs_starts() says so */
  float xai_temperature_len;    /* > 0: logits of a query at position p > len are multiplied by
                                   log2(p) / log2(len) (:171-177); 0 => off.  With soft_cap set as well
                                   the factor multiplies the capped logit, the order of
                                   ref_ragged_paged_attention (:166-177); the reference's TPU kernel
                                   multiplies first and caps after (:481-486), so the reference's two
                                   paths differ from each other when both options are on */
  int32_t mask_mode;            /* RpaMaskMode */
  int32_t mask_rows_page_aligned; /* custom mask row_width_i: 0 => kv_len_i, 1 => kv_len_i rounded up to
                                   pages (cu_kv_lens delta; mask_aligned_to_cu_kv, :1791-1806) */
  int32_t softmax_dtype;        /* RpaSoftmaxDtype: the masked logits (and the sink) are rounded to this type
                                   before the softmax (:181-186, kernel :522-523); maxima, exponentials and
                                   sums stay f32 */
  float q_scale;                /* > 0: queries are divided by it and rounded to the cache's element type
                                   (fp8 saturating at +-448) before the first product, the logits multiplied
                                   by it (kernel :463-478); 0 => off */
  /* ---- static-shape mode: the batch composition read on the device ----
   * Device i32[3] (decode_end, prefill_end, num_seqs) as ragged_paged_attention takes it
   * (ragged_paged_attention_v3.py:1676, dispatch :2060-2090), or NULL.  When given, the host fields
   * decode_end and sum_decode_kv_len are ignored and num_seqs is only the static bound S (the length of
   * kv_lens): grids are sized from T, S and the page-table bound, every workgroup reads the
   * composition itself and the ones with nothing to do leave at once, so one compiled call serves
   * every batch of a bucket and nothing is read back to the host.  128- and 256-wide heads alike.
   * Neither mode limits the sequences or tokens of a call beyond int32: rows are folded onto the first
   * grid dimension. */
  const int32_t* distribution;
  /* ---- read only with RPA_PARAMS_TAIL in `layout` ---- */
  /* Elements of a row of q, out, keys and values where that is less than the cache's head_dim (the reference pads heads
   * to a multiple of 128, rpa_v3:1187-1241): a multiple of 8 (e4m3: 16), head_dim - q_head_dim < 128; 0 = head_dim.
   * The rest of a cached row is zero, is written as zeros with the new tokens and adds nothing. */
  int32_t q_head_dim;
  /* 1: no sequence of the call has tokens in the cache before its new ones (kv_len == query tokens, known on the host).
   * rpa_attention_update then attends to the keys / values it is given and fills the cache beside that. */
  int32_t prompts_only;
} RpaParams;

/*
 * Absorbed-MLA decode (mla_ragged_paged_attention, kernels/mla/v2/kernel.py:1338-1370;
 * oracle ref_mla_ragged_paged_attention, kernels/mla/v1/ref.py:108-248).
 * One shared latent row per token: [kv_c (lkv_dim) | k_pe (rope_dim)], rows of
 * `row_stride` elements (576 compact, 640 in the reference's 128-aligned layout
 * with rope at element offset `rope_offset`).
 */
typedef struct RpaMlaParams {
  const void* ql_nope;        /* bf16 [T, Hq, lkv_dim] */
  const void* q_pe;           /* bf16 [T, Hq, rope_dim] */
  void* out;                  /* bf16 [T, Hq, lkv_dim] */
  const void* cache_kv;       /* bf16 (or fp8-e4m3, see cache_dtype) [pages, P, row_stride] */
  const int32_t* kv_lens;
  const int32_t* page_indices;
  const int32_t* cu_q_lens;
  const int32_t* cu_kv_lens;  /* NULL => padded table with pages_per_seq stride */
  void* workspace;
  size_t workspace_bytes;
  int32_t num_tokens;
  int32_t num_seqs;           /* rpa_mla_decode: all must be decode rows (q_len == 1) */
  int32_t num_q_heads;
  int32_t lkv_dim;            /* 512 */
  int32_t rope_dim;           /* 64 */
  int32_t row_stride;         /* elements per cached token row */
  int32_t rope_offset;        /* element offset of k_pe inside a row */
  int32_t page_size;
  int32_t total_pages;
  int32_t pages_per_seq;
  int32_t max_kv_len;
  int32_t num_splits;         /* 0 => automatic */
  int32_t sliding_window;     /* 0 => off */
  float sm_scale;
  float soft_cap;             /* 0 => off */
  float mask_value;           /* 0 => default */
  int64_t sum_kv_len;         /* what the call's rows see, added up (host-side, the plans go by it); 0 => unknown: the kv_lens of
                                 decode rows, of chunks what every query token sees */
  /* Scalar scales of kernels/mla/v2/kernel.py:1354-1356 (used at :372-375, :408-409; oracle
   * kernels/mla/v1/ref.py:223-226, 241-242): logits are multiplied by k_scale and q_scale next to
   * sm_scale, the output by v_scale.  0 => off. */
  float q_scale;
  float k_scale;
  float v_scale;
  /* Static-shape mode (see RpaParams.distribution): device i32[3] or NULL.  When given, num_seqs is
   * the static bound and rpa_mla_attention / rpa_mla_kv_write read distribution[2] on the device;
   * rpa_mla_decode (decode rows known on the host) does not take it. */
  const int32_t* distribution;
  /* Element type of cache_kv (and of the rows rpa_mla_kv_write takes): RPA_KV_BF16 (0, the default) or
   * RPA_KV_FP8_E4M3 -- latent rows of one byte per element, expanded to bf16 on their way through
   * LDS; k_scale / v_scale above are their dequantisation scales (kernels/mla/v1/ref.py:223-226,
   * 241-242).  row_stride and rope_offset stay in elements (multiples of 16 for fp8). */
  int32_t cache_dtype;
  int32_t reserved0;
} RpaMlaParams;

/* Library version (RPA_VERSION of the build). */
RPA_API int rpa_version(void);

/* Thread-local description of the last error returned on this thread. */
RPA_API const char* rpa_last_error(void);

/*
 * Static contract check: static_validate_inputs,
 * ragged_paged_attention_v3.py:1314-1439 (3-D q, Hq % Hkv == 0,
 * sliding_window > 0, soft_cap != 0, ...).  Called by every entry point.
 */
RPA_API int rpa_validate(const RpaParams* p);

/*
 * Value check on HOST copies of the metadata: dynamic_validate_inputs,
 * ragged_paged_attention_v3.py:1442-1487 (0 < q_len <= kv_len, page count and
 * page index ranges, distribution ordering).  Pointers are host memory.
 */
RPA_API int rpa_validate_host(const RpaParams* p, const int32_t* kv_lens, const int32_t* page_indices,
                      int64_t num_page_indices, const int32_t* cu_q_lens,
                      const int32_t* cu_kv_lens, const int32_t* distribution);

/*
 * Bytes of workspace for `p`: what the decode rows' split-KV plan needs (rpa_decode fails without
 * it), or, if larger, the room that lets a prefill launch which would leave most of the GPU idle
 * (one long prompt on a few heads, a verify step on a long context) cut its K/V ranges into pieces
 * and merge them, and that holds a custom mask as one bit per (query token, kv token); rpa_prefill uses
 * that room when it is there and otherwise runs whole ranges and reads the mask's i32 words (slower,
 * same results to the tolerance of the path).  Two plans of the decode rows ask for room that they can do
 * without: rows of one length whose even pieces would leave most of a last round of the GPU empty (from
 * 256 MB on whole rows too), and small batches of 256-wide heads.  With less than this function reports, they
 * run on the plan that needs less, or nothing: slower, same results to the tolerance of the path.
 */
RPA_API size_t rpa_workspace_bytes(const RpaParams* p);
RPA_API size_t rpa_mla_workspace_bytes(const RpaMlaParams* p);

/*
 * Page-table gather of one sequence (the indexing expression
 * k_pages[page_indices[i]].reshape(-1, Hkv, D)[:kv_len] of
 * ragged_paged_attention_v3.py:138-139).  Copies, bit for bit, the K rows and
 * V rows of sequence `seq` into k_out / v_out [kv_len, Hkv, D] (kv dtype).
 */
RPA_API int rpa_gather_pages(const RpaParams* p, int32_t seq, void* k_out, void* v_out,
                     int32_t max_tokens, void* stream);

/*
 * Decode rows [0, decode_end): split-KV pass + combine pass.  Stands in for the
 * DECODE pallas_call of ragged_paged_attention_v3.py:2065-2072.
 */
RPA_API int rpa_decode(const RpaParams* p, void* stream);

/*
 * Prefill / mixed rows [decode_end, num_seqs): flash-style MFMA kernel.  Stands
 * in for the PREFILL and MIXED pallas_calls, ragged_paged_attention_v3.py:2074-2090.
 */
RPA_API int rpa_prefill(const RpaParams* p, void* stream);

/*
 * Whole call: dispatch by distribution exactly as
 * ragged_paged_attention_v3.py:2060-2090 does (decode rows, then the rest).
 */
RPA_API int rpa_attention(const RpaParams* p, void* stream);

/*
 * Which launch shape a call would take, as text: the row of the library's shape table (kernel family, query
 * positions x query heads x K/V tokens per workgroup, waves walked together, resident waves), the split plan
 * of the decode rows and the workspace behind it, whether a prefill launch takes its sequences one after the other, and
 * who leaves the new tokens of rpa_attention_update in the cache.
 * "whole call" stands in front where rpa_attention and rpa_attention_update run every query token as a row of the decode
 * kernels (few tokens on short contexts, workspace of rpa_workspace_bytes()); "decode" and "prefill" are then what
 * rpa_decode and rpa_prefill take.  The counterpart of the reference's get_tuned_block_sizes /
 * get_default_block_sizes, which answer the same question for its tile table
 * (kernels/ragged_paged_attention/tuned_block_sizes_v3.py:2163-2229, ragged_paged_attention_v3.py:1490-1638).
 * Host arithmetic only (no launch, no device read).  Writes at most len - 1 characters plus a NUL into buf and
 * returns the length of the whole text (as snprintf does), or a negative RpaStatus.  The plan is the one that a call with
 * rpa_workspace_bytes() of workspace takes, whatever p->workspace says.
 */
RPA_API int rpa_describe_plan(const RpaParams* p, char* buf, size_t len);

/*
 * rpa_attention for callers that cannot allocate device memory (code under HIP graph capture,
 * tight serving loops, harnesses that forbid it).  No counterpart in the reference, where XLA owns
 * every buffer.  Same arguments and results as rpa_attention, except that p->workspace and
 * p->workspace_bytes are ignored: the split-KV workspace is an array the library holds itself on
 * every GPU, rpa_noalloc_max_workspace_bytes() (40 MiB) long.  A batch whose decode rows need more
 * than that is refused with RPA_EINVAL_WORKSPACE; a prefill launch that would cut its K/V ranges
 * does so only if its partial rows fit the array (otherwise it runs whole ranges: the same rows to
 * the tolerance of the path, not bit for bit).  The call allocates and frees nothing.  All
 * calls on one GPU share the array: calls that overlap on one GPU (two streams, a graph replay next
 * to eager work) race on it; order them on one stream.
 */
RPA_API size_t rpa_noalloc_max_workspace_bytes(void);
RPA_API int rpa_attention_noalloc(const RpaParams* p, void* stream);

/*
 * Scatter the new K/V rows of every sequence into the paged cache: the fused
 * cache update of ragged_paged_attention_v3.py:670-719 / the standalone
 * kv_cache_update of kernels/update_kv_cache/update_kv_cache.py:120.  Token j of
 * sequence i goes to position kv_len_i - q_len_i + j.  keys/values are
 * [T, Hkv, D] in the cache dtype.
 */
RPA_API int rpa_kv_write(const RpaParams* p, const void* keys, const void* values, void* stream);

/*
 * rpa_kv_write and rpa_attention as one call: ragged_paged_attention as the reference's layers call it
 * (ragged_paged_attention_v3.py:1667-2097 writes the new tokens and attends to them in one kernel).  keys / values:
 * [T, Hkv, D] in the cache dtype, or both NULL when the cache already holds every token.
 *
 * Every sequence sees its own new tokens.  Whether it sees those that another sequence of the same call brings into a page that
 * both tables name is not defined: the cache is written in front of the attention, beside it or by it, by what the call is.  A call
 * behind this one on the stream finds all of them.
 */
RPA_API int rpa_attention_update(const RpaParams* p, const void* keys, const void* values, void* stream);

/* n words of host memory to device memory in stream order (a batch's metadata); the source may be reused at once, the
 * destination is whole once the stream has come that far: work on other streams waits for an event behind it. */
RPA_API int rpa_upload_words(int32_t* dst, const int32_t* src, int32_t n, void* stream);

/* Whether a RPA_MASK_CUSTOM call needs cu_mask_lens: 0 where the mask is turned into bits first (128-wide heads, max_kv_len
 * given, rpa_workspace_bytes() of workspace), which finds the starts of the sequences' rows by itself. */
RPA_API int rpa_mask_needs_starts(const RpaParams* p);

/* Absorbed-MLA decode, see RpaMlaParams: every sequence contributes exactly one query token. */
RPA_API int rpa_mla_decode(const RpaMlaParams* p, void* stream);

/*
 * Absorbed-MLA attention for any batch composition (decode, prefill chunks, mixed): the three
 * launches of mla_ragged_paged_attention (kernels/mla/v2/kernel.py:1338-1744) in one.  Query
 * token j of a sequence with q_len new tokens attends to the cache tokens 0 .. kv_len - q_len + j.
 * Workspace: rpa_mla_attention_workspace_bytes(); max_kv_len / sum_kv_len bound, resp. sum, the
 * per-token visible lengths.
 */
RPA_API size_t rpa_mla_attention_workspace_bytes(const RpaMlaParams* p);
RPA_API int rpa_mla_attention(const RpaMlaParams* p, void* stream);

/* rpa_describe_plan for the absorbed-MLA entry points: token_rows = 0 describes rpa_mla_decode, 1 rpa_mla_attention. */
RPA_API int rpa_mla_describe_plan(const RpaMlaParams* p, int token_rows, char* buf, size_t len);

/*
 * Write the new latent rows into the paged cache: update_kv_cache of kernels/mla/v1/ref.py:56-105
 * (the fused cache update of kernels/mla/v2/kernel.py).  new_kv_c bf16 [T, lkv_dim], new_k_pe bf16
 * [T, rope_dim]; token j of sequence i goes to position kv_len_i - q_len_i + j.
 */
RPA_API int rpa_mla_kv_write(const RpaMlaParams* p, const void* new_kv_c, const void* new_k_pe, void* stream);

/*
 * rpa_mla_kv_write and rpa_mla_decode (token_rows = 0) or rpa_mla_attention (token_rows = 1) as one call; the new rows
 * may both be NULL when the cache already holds every token.  New tokens in pages of several sequences: as
 * rpa_attention_update has it.
 */
RPA_API int rpa_mla_attention_update(const RpaMlaParams* p, const void* new_kv_c, const void* new_k_pe, int token_rows,
                             void* stream);

/*
 * Sparse absorbed-MLA attention (kernels/dsa/sparse_mla.py:63-297): every query token attends to its own selection of
 * its sequence's cached tokens, as if it were a decode row over a page table of the selection.
 *   k_pages_max > 0   whole pages (sparse_mla.py:63-203, decode rows): the distinct pages the selection touches, ascending,
 *                     at most k_pages_max - 1 of them, then the page of the new token, into which the new row is written.
 *                     The last page of the cache is the padding target.
 *   k_pages_max == 0  single tokens (sparse_mla.py:206-297): the valid entries of the selection, which come first; the
 *                     new row stands for the last of them and the cache is not written.
 * `p` is the batch as rpa_mla_decode takes it (ragged page table; kv_lens, cu_q_lens of num_seqs sequences; max_kv_len
 * and sum_kv_len are not read; sliding_window counts tokens of the selection).  The new rows may both be NULL when the
 * cache already holds every token.
 */
typedef struct RpaMlaSparse {
  const int32_t* topk;       /* i32[T, topk_stride]: positions in the sequence, -1 = unused */
  int32_t topk_count;        /* entries of a row that are read */
  int32_t topk_stride;
  int32_t topk_is_pages;     /* whole pages: the entries are pages of the sequence already */
  int32_t pages_per_seq;
  int32_t k_pages_max;
  int32_t num_page_indices;  /* entries of p->page_indices */
} RpaMlaSparse;
RPA_API size_t rpa_mla_sparse_workspace_bytes(const RpaMlaParams* p, const RpaMlaSparse* s);
RPA_API int rpa_mla_sparse_attention(const RpaMlaParams* p, const RpaMlaSparse* s, const void* new_kv_c,
                                     const void* new_k_pe, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* RPA_MI355_H_ */
