"""The work that users of this package have it do, as cases that can be timed and compared.

A case is one pass through the public entry points: a layer call of the attention backends, a whole decode step
(metadata and every layer), or a call of one of the functional operators.  Lengths and the composition of a batch
follow from the case alone; values, page placement and selections follow from the seed.  ``kind`` says how a program
calls the package:

* ``layer``   ``FlashAttention`` layer calls on metadata built before (a forward pass builds it once)
* ``step``    ``get_forward_metadata`` and then one call per layer: the attention of a whole forward pass
* ``call``    ``ragged_paged_attention`` with a host composition: decode rows, chunks, or both in one batch
* ``bucket``  ``ragged_paged_attention`` with the composition on the device, batch and tokens padded to a bucket
* ``verify``  ``ragged_paged_attention`` on a flat tree mask, as speculative decoding verifies its drafts
* ``mla``     ``MLAAttentionBackend`` layer call (bf16 latents) or ``mla_ragged_paged_attention`` (e4m3 latents)
* ``sparse``  ``sparse_mla_page_level`` / ``sparse_mla_via_dense`` on the rows that an indexer selected

Every call brings the new tokens with it: they are written into the paged cache, then attended to.
"""

import math
from types import SimpleNamespace

import numpy as np
import torch

from __graft_entry__ import load_package

pkg = load_package()
DEV = torch.device("cuda:0")
LATENT, ROPE = 512, 64


# ---------------------------------------------------------------------------------------------- the cases
def _gqa(kind, **kw):
    """seqs decode rows or chunks; `chunks` more chunks behind the decode rows of a mixed batch."""
    c = dict(kind=kind, seqs=1, new_lo=1, new_hi=1, old_lo=0, old_hi=0, chunks=0, chunk_lo=0, chunk_hi=0, chunk_old_hi=0,
             heads=32, kv_heads=8, head_dim=128, page=64, dtype="bf16", window=0, cap=0.0, sink=False, layers=1)
    c.update(kw)
    return c


def _mla(kind, **kw):
    c = dict(kind=kind, seqs=1, new_lo=1, new_hi=1, old_lo=0, old_hi=0, heads=128, width=LATENT + ROPE, page=64,
             dtype="bf16")
    c.update(kw)
    return c


def listed():
    return [
        # a handful of requests decoding on a small model whose step is one compiled call for every batch of the
        # bucket: 5 requests in a bucket of 8, a few hundred cached tokens, 16-token pages.  Latency is all there is.
        _gqa("bucket", name="decode_bucket_small", seqs=5, old_lo=63, old_hi=511, heads=16, kv_heads=8, page=16),
        # the attention of one whole decode step of Qwen3-0.6B (28 layers, 16 / 8 heads) for 8 chat requests
        _gqa("step", name="decode_step_28_layers", seqs=8, old_lo=63, old_hi=511, heads=16, kv_heads=8, page=16,
             layers=28),
        # a loaded server on a tensor-parallel shard (8 / 4 heads, 128-token pages): 128 requests of 1-2 k tokens
        _gqa("layer", name="decode_128_rows_tp_shard", seqs=128, old_lo=1024, old_hi=2047, heads=8, kv_heads=4, page=128),
        # Llama-3-8B, continuous batching with chunked prefill: 56 decode rows and 8 chunks in one call
        _gqa("call", name="mixed_decode_and_chunks", seqs=56, old_lo=511, old_hi=4095, chunks=8, chunk_lo=128,
             chunk_hi=2048, chunk_old_hi=2048),
        # Llama-3-8B on long documents: 16 rows of 32 k tokens, the most cache a decode call reads here
        _gqa("layer", name="decode_long_context", seqs=16, old_lo=32767, old_hi=32767),
        # Qwen3-32B on an e4m3 cache, a full layer and a 4096-token sliding-window layer one after the other
        _gqa("call", name="decode_e4m3_full_and_window", seqs=128, old_lo=1023, old_hi=8191, heads=64, dtype="e4m3",
             window=4096, layers=2),
        # time to first token of one prompt of odd length on a tensor-parallel shard
        _gqa("layer", name="prompt_1000_tokens_tp_shard", new_lo=1003, new_hi=1003, heads=8, kv_heads=2),
        # Llama-3-8B, long prompts in chunks of 2048 on prefixes of up to 16 k tokens: the matrix work of a prefill server
        _gqa("layer", name="chunked_prefill_long", seqs=4, new_lo=1900, new_hi=2048, old_lo=4096, old_hi=16384),
        # prompts on a model with 256-wide heads, logit soft cap and a sliding window on an e4m3 cache
        _gqa("call", name="prefill_wide_heads_cap_e4m3", seqs=6, new_lo=300, new_hi=1500, old_lo=0, old_hi=3000, heads=16,
             kv_heads=8, head_dim=256, dtype="e4m3", window=1024, cap=50.0),
        # DeepSeek-V3 decode on the latent cache, all 128 heads on one GPU
        _mla("mla", name="mla_decode_128_heads", seqs=64, old_lo=2047, old_hi=16383),
        # DeepSeek-V3 prefill chunks of 512 tokens on 4 k prefixes, reference's 640-wide latent rows
        _mla("mla", name="mla_prefill_128_heads", seqs=4, new_lo=512, new_hi=512, old_lo=4096, old_hi=4096, width=640),
        # DeepSeek sparse attention while decoding: whole pages that the indexer's 2048 best tokens touch, 16 heads
        _mla("sparse", name="sparse_mla_decode_pages", seqs=32, old_lo=2047, old_hi=32767, heads=16, width=640,
             level="page", topk=2048, kp=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _span(rng, lo, hi):
    """Bounds of a batch's lengths: anywhere in the range, from equal lengths to very ragged ones."""
    a, b = sorted((_log(rng, lo, hi), _log(rng, lo, hi)))
    return a, b


def _draw_once(rng):
    kind = rng.choice(["bucket", "step", "layer", "layer", "layer", "call", "call", "call", "verify", "mla", "mla", "mla",
                       "sparse", "sparse"])
    if kind in ("mla", "sparse"):
        heads, page = rng.choice([16, 32, 64, 128]), rng.choice([16, 64, 128])
        width = rng.choice([576, 640])
        if kind == "sparse":
            lo, hi = _span(rng, 300, 32767)
            return _mla("sparse", seqs=_log(rng, 1, 64), old_lo=lo, old_hi=hi, heads=heads, page=page, width=width,
                        level=rng.choice(["page", "token"]), topk=rng.choice([512, 1024, 2048]), kp=64)
        dtype = rng.choice(["bf16", "bf16", "e4m3"])
        if rng.random() < 0.5:
            lo, hi = _span(rng, 100, 16383)
            return _mla("mla", seqs=_log(rng, 1, 128), old_lo=lo, old_hi=hi, heads=heads, page=page, width=width, dtype=dtype)
        n_lo, n_hi = _span(rng, 16, 2048)
        return _mla("mla", seqs=_log(rng, 1, 8), new_lo=n_lo, new_hi=n_hi, old_lo=0, old_hi=_log(rng, 64, 8192), heads=heads,
                    page=page, width=width, dtype=dtype)
    heads, kv_heads = rng.choice([(8, 1), (8, 2), (8, 4), (16, 8), (32, 8), (40, 8), (64, 8)])
    page = rng.choice([16, 64, 64, 128])
    if kind == "bucket":
        lo, hi = _span(rng, 30, 8000)
        return _gqa("bucket", seqs=_log(rng, 1, 128), old_lo=lo, old_hi=hi, heads=heads, kv_heads=kv_heads, page=page)
    if kind == "step":
        lo, hi = _span(rng, 30, 2000)
        return _gqa("step", seqs=_log(rng, 1, 8), old_lo=lo, old_hi=hi, heads=16, kv_heads=rng.choice([2, 4, 8]), page=page,
                    layers=rng.randint(2, 24))
    if kind == "verify":
        lo, hi = _span(rng, 100, 16000)
        n = rng.choice([4, 8, 16])
        return _gqa("verify", seqs=_log(rng, 1, 32), new_lo=n, new_hi=n, old_lo=lo, old_hi=hi, heads=heads, kv_heads=kv_heads,
                    page=page)
    o = dict(heads=heads, kv_heads=kv_heads, page=page)
    if kind == "call":
        o["dtype"] = rng.choice(["bf16", "e4m3"])
        o["window"] = rng.choice([0, 0, 512, 4096])
        o["cap"] = rng.choice([0.0, 0.0, 0.0, 30.0])
        if rng.random() < 0.25:
            o.update(head_dim=256, heads=16, kv_heads=rng.choice([2, 4, 8]))
    else:
        o["window"] = rng.choice([0, 0, 0, 1024])
        o["sink"] = rng.random() < 0.15
        o["head_dim"] = rng.choice([128, 128, 128, 64])
    shape = rng.choice(["decode", "decode", "prefill", "mixed" if kind == "call" else "prefill"])
    if shape == "decode":
        lo, hi = _span(rng, 60, 32767)
        return _gqa(kind, seqs=_log(rng, 1, 256), old_lo=lo, old_hi=hi, **o)
    n_lo, n_hi = _span(rng, 16, 4096)
    old_hi = rng.choice([0, _log(rng, 100, 16384)])
    if shape == "prefill":
        return _gqa(kind, seqs=_log(rng, 1, 8), new_lo=n_lo, new_hi=n_hi, old_lo=0, old_hi=old_hi, **o)
    lo, hi = _span(rng, 60, 8000)
    return _gqa(kind, seqs=_log(rng, 1, 64), old_lo=lo, old_hi=hi, chunks=_log(rng, 1, 8), chunk_lo=n_lo, chunk_hi=n_hi,
                chunk_old_hi=old_hi, **o)


def draw(rng):
    """A case of the same ranges; what would read more than the long-context decode case or multiply more than a
    third of the largest prefill case is drawn again."""
    while True:
        c = _draw_once(rng)
        w = work(c)
        if w["bytes"] < 2.2e9 and w["flops"] < 8e11:
            return c


# ---------------------------------------------------------------------------------------------- their sizes
def _lengths(c):
    """(new tokens, cached tokens) per sequence: decode rows first, then chunks."""
    rng = np.random.default_rng([c["seqs"], c["new_lo"], c["new_hi"], c["old_lo"], c["old_hi"], c.get("chunks", 0)])
    new = rng.integers(c["new_lo"], c["new_hi"], size=c["seqs"], endpoint=True)
    old = rng.integers(c["old_lo"], c["old_hi"], size=c["seqs"], endpoint=True)
    if c.get("chunks"):
        new = np.concatenate([new, rng.integers(c["chunk_lo"], c["chunk_hi"], size=c["chunks"], endpoint=True)])
        old = np.concatenate([old, rng.integers(0, c["chunk_old_hi"], size=c["chunks"], endpoint=True)])
    return new.astype(np.int64), old.astype(np.int64)


def _windows(c):
    """The window of each layer: where a case has several layers and a window, every other one has it."""
    return [c["window"] if c["layers"] == 1 or i % 2 else 0 for i in range(c["layers"])]


def work(c):
    new, old = _lengths(c)
    T, kv = int(new.sum()), new + old
    meta = 4 * int((-(-kv // c["page"])).sum() + 3 * len(kv))
    if c["kind"] in ("mla", "sparse"):
        H, size = c["heads"], 1 if c["dtype"] == "e4m3" else 2
        row = (LATENT + ROPE) * size
        if c["kind"] == "sparse":
            rows = np.minimum(kv, c["topk"] if c["level"] == "token" else c["kp"] * c["page"])
            read, pairs = int(rows.sum()), int(rows.sum())
            meta += 4 * T * c["topk"]
        else:
            read, pairs = int(old.sum()), int((new * old + new * (new + 1) // 2).sum())
        io = T * H * (2 * LATENT + ROPE) * 2
        wrote = T * row * (1 if c["kind"] == "sparse" and c["level"] == "token" else 2)
        return {"bytes": read * row + wrote + io + meta, "flops": pairs * H * (4 * LATENT + 2 * ROPE)}
    H, K, D = c["heads"], c["kv_heads"], c["head_dim"]
    token = 2 * K * D * (1 if c["dtype"] == "e4m3" else 2)
    nbytes = flops = 0
    for w in _windows(c):
        seen = np.minimum(old, np.maximum(w - 1, 0)) if w else old
        nbytes += int(seen.sum()) * token + T * token * 2 + 2 * T * H * D * 2 + meta
        if c["kind"] == "verify":
            nbytes += 4 * int((new * kv).sum())
        for n, o in zip(new.tolist(), old.tolist()):
            if c["kind"] == "verify":
                pairs = n * (n + o)
            elif w:
                pairs = int(np.minimum(o + 1 + np.arange(n), w).sum())
            else:
                pairs = n * o + n * (n + 1) // 2
            flops += 4 * H * D * pairs
    return {"bytes": nbytes, "flops": flops}


def tolerance(c):
    # bf16 operands, probabilities and results (2^-9 each), sums in 32 bits
    return {"rel": 1e-2}


# ---------------------------------------------------------------------------------------------- their inputs
class _Inputs:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)
        self.rng = np.random.default_rng(seed)

    def normal(self, *shape, std=1.0, dtype=torch.bfloat16):
        out = torch.empty(shape, dtype=dtype, device=DEV)
        flat = out.view(-1)
        for s in range(0, flat.numel(), 1 << 27):  # in slabs: the wide draw stays small beside the pool
            e = min(flat.numel(), s + (1 << 27))
            flat[s:e] = (torch.randn(e - s, generator=self.g, device=DEV, dtype=torch.bfloat16) * std).clamp(-448, 448).to(dtype)
        return out

    def pages(self, kv, page):
        """Physical pages of every sequence, scattered over a pool with a few pages to spare."""
        counts = -(-kv // page)
        total = int(counts.sum())
        return self.rng.permutation(total + 3)[:total].astype(np.int32), total + 3

    def up(self, a, dtype=np.int32):
        return torch.from_numpy(np.ascontiguousarray(a, dtype=dtype)).to(DEV)


def _cumsum(x):
    return np.concatenate([[0], np.cumsum(x)]).astype(np.int32)


def _batch(c, new, kv, pages):
    """What the scheduler hands to the backend: slots of every sequence's pages, one after the other."""
    mode = pkg.ForwardMode.DECODE if c["new_hi"] == 1 else pkg.ForwardMode.EXTEND
    loc = (pages.astype(np.int64)[:, None] * c["page"] + np.arange(c["page"])).reshape(-1).astype(np.int32)
    return SimpleNamespace(forward_mode=mode, seq_lens=kv.astype(np.int32), cache_loc=loc,
                           extend_seq_lens=new.astype(np.int32), dp_size=1, per_dp_bs_size=len(kv))


class _Pool:
    """The engine's cache: one fused buffer per layer out of one allocation."""

    def __init__(self, all_layers):
        self.all_layers = all_layers
        self.layers = list(all_layers.unbind(0))

    def get_fused_kv_buffer(self, layer_id):
        return self.layers[layer_id]


def _bytes(cache):
    return cache.view(torch.uint8) if cache.dtype == torch.float8_e4m3fn else cache


def _prepare_gqa(c, seed):
    x = _Inputs(seed)
    new, old = _lengths(c)
    kv, T, L = new + old, int(new.sum()), c["layers"]
    H, K, D = c["heads"], c["kv_heads"], c["head_dim"]
    pages, pool_pages = x.pages(kv, c["page"])
    e4m3 = c["dtype"] == "e4m3"
    dt = torch.float8_e4m3fn if e4m3 else torch.bfloat16
    # rows of the pool are stored at a multiple of 128; e4m3 rows spread over the type's range, per-head scales undo it
    wide = -(-D // 128) * 128
    std = 64.0 if e4m3 else 1.0
    cache = x.normal(L, pool_pages, c["page"], 2 * K, wide, std=std, dtype=dt)
    if wide != D:
        cache[..., D:] = 0
    s = SimpleNamespace(c=c, new=new, kv=kv, T=T, cache=cache, pool=_Pool(cache), out_cache=_bytes(cache))
    pad = T
    if c["kind"] == "bucket":
        pad = 1 << (T - 1).bit_length() if T > 4 else 4
    # logits of a few units, as trained models have them
    s.q = [x.normal(pad, H, D, std=2.0) for _ in range(L)]
    s.k = [x.normal(pad, K, D, std=std, dtype=dt) for _ in range(L)]
    s.v = [x.normal(pad, K, D, std=std, dtype=dt) for _ in range(L)]
    s.scale = D ** -0.5
    s.opts = dict(sm_scale=s.scale, soft_cap=c["cap"] or None)
    if e4m3:
        s.opts.update(k_scale=torch.rand(K, generator=x.g, device=DEV) * 0.005 + 0.01,
                      v_scale=torch.rand(K, generator=x.g, device=DEV) * 0.005 + 0.01)
    s.sink = torch.randn(H, generator=x.g, device=DEV) if c["sink"] else None
    s.windows = [w or None for w in _windows(c)]
    if c["kind"] in ("layer", "step"):
        s.batch = _batch(c, new, kv, pages)
        s.backend = pkg.FlashAttention(H, K, D, page_size=c["page"], device=DEV)
        s.layers = [SimpleNamespace(layer_id=i, scaling=s.scale, head_dim=D, sliding_window_size=w, logit_cap=c["cap"],
                                    xai_temperature_len=-1, softmax_dtype=None, attn_type=None)
                    for i, w in enumerate(s.windows)]
        s.backend.forward_metadata = s.backend.get_forward_metadata(s.batch)
        s.q, s.k, s.v = ([t.view(pad, -1) for t in ts] for ts in (s.q, s.k, s.v))
        return s
    n, lens = len(kv), kv
    decode = int(n - c["chunks"]) if c["new_hi"] == 1 else 0
    if c["kind"] == "bucket":
        lens = np.concatenate([kv, np.zeros(pad - n, dtype=np.int64)])
        new = np.concatenate([new, np.zeros(pad - n, dtype=np.int64)])
    s.kv_lens, s.pages = x.up(lens), x.up(pages)
    s.cu_q, s.cu_kv = x.up(_cumsum(new)), x.up(_cumsum(-(-lens // c["page"]) * c["page"]))
    s.dist = np.array([decode, decode, n], dtype=np.int32)
    if c["kind"] == "bucket":
        s.dist = x.up(s.dist)
        s.opts.update(max_kv_len=1 << int(kv.max() - 1).bit_length())
    else:
        chunks = new[decode:]
        s.opts.update(max_kv_len=int(kv.max()), max_q_len=int(chunks.max()) if len(chunks) else 1,
                      host_kv_lens=kv.astype(np.int32))
    s.mask = None
    if c["kind"] == "verify":
        # every draft token sees the prefix, itself and some of the drafts before it
        d = c["new_hi"]
        rows = []
        for o in old.tolist():
            tree = np.tril(x.rng.random((d, d)) < 0.5).astype(np.int32)
            np.fill_diagonal(tree, 1)
            rows.append(np.concatenate([np.ones((d, o), dtype=np.int32), tree], axis=1).reshape(-1))
        md = pkg.build_verify_metadata(seq_lens=old.astype(np.int32), draft_token_num=d, logits_indices_selector=np.arange(n),
                                       custom_mask=np.concatenate(rows), page_size=c["page"])
        s.mask = x.up(md["custom_mask"])
        s.opts.update(causal=0, mask_aligned_to_cu_kv=True)
    return s


def _prepare_mla(c, seed):
    x = _Inputs(seed)
    new, old = _lengths(c)
    kv, T, H = new + old, int(new.sum()), c["heads"]
    pages, pool_pages = x.pages(kv, c["page"])
    dt = torch.float8_e4m3fn if c["dtype"] == "e4m3" else torch.bfloat16
    std = 20.0 if c["dtype"] == "e4m3" else 0.5
    cache = x.normal(pool_pages, c["page"], c["width"], std=std, dtype=dt)
    s = SimpleNamespace(c=c, cache=cache, out_cache=_bytes(cache))
    s.q, s.q_rope = x.normal(T, H, LATENT, std=0.5), x.normal(T, H, ROPE, std=0.5)
    s.k, s.k_rope = x.normal(T, LATENT, std=std, dtype=dt), x.normal(T, ROPE, std=std, dtype=dt)
    s.scale = 192 ** -0.5
    if c["kind"] == "mla" and c["dtype"] == "bf16":
        s.pool = SimpleNamespace(get_fused_kv_buffer=lambda layer_id: cache)
        s.layer = SimpleNamespace(layer_id=0, scaling=s.scale, sliding_window_size=None, logit_cap=None)
        s.backend = pkg.MLAAttentionBackend(H, LATENT, 128, ROPE, 128, page_size=c["page"], device=DEV)
        s.batch = _batch(c, new, kv, pages)
        s.backend.forward_metadata = s.backend.get_forward_metadata(s.batch)
        return s
    n = len(kv)
    s.kv_lens, s.pages, s.cu_q = x.up(kv), x.up(pages), x.up(_cumsum(new))
    s.cu_kv = x.up(_cumsum(-(-kv // c["page"]) * c["page"]))
    s.dist = np.array([n, n, n] if c["new_hi"] == 1 else [0, 0, n], dtype=np.int32)
    if c["kind"] == "mla":
        s.opts = dict(k_scale=0.025, v_scale=0.025, max_kv_len=int(kv.max()),
                      sum_kv_len=int((new * kv - new * (new - 1) // 2).sum()))
        return s
    # the indexer's choice: the best-scored cached tokens, close together more often than not, the newest one last
    lens = torch.from_numpy(kv).to(DEV)
    most, k = int(kv.max()), c["topk"]
    near = torch.rand(n, -(-most // 64), generator=x.g, device=DEV).repeat_interleave(64, dim=1)[:, :most]
    score = near + torch.rand(n, most, generator=x.g, device=DEV)
    at = torch.arange(most, device=DEV)[None, :]
    score = torch.where(at < lens[:, None] - 1, score, torch.full_like(score, -1.0))
    m = min(k - 1, most)
    best = score.topk(m, dim=1)
    idx = torch.full((n, k), -1, dtype=torch.int64, device=DEV)
    idx[:, :m] = torch.where(best.values >= 0, best.indices, torch.full_like(best.indices, -1))
    last = torch.clamp(lens - 1, max=k - 1)
    idx.scatter_(1, last[:, None], (lens - 1)[:, None])
    s.topk = idx.to(torch.int32).contiguous()
    s.pages_per_seq = -(-most // c["page"])
    return s


def prepare(case, seed):
    return _prepare_mla(case, seed) if case["kind"] in ("mla", "sparse") else _prepare_gqa(case, seed)


# ---------------------------------------------------------------------------------------------- one pass
def run(s):
    c = s.c
    if c["kind"] in ("layer", "step"):
        if c["kind"] == "step":
            s.backend.forward_metadata = s.backend.get_forward_metadata(s.batch)
        outs = []
        for layer, q, k, v in zip(s.layers, s.q, s.k, s.v):
            o, _ = s.backend(q, k, v, layer, s.batch, s.pool, attention_sink=s.sink)
            outs.append(o)
        return outs, s.out_cache
    if c["kind"] in ("call", "bucket", "verify"):
        outs = []
        for i, window in enumerate(s.windows):
            o, _ = pkg.ragged_paged_attention(s.q[i], s.k[i], s.v[i], s.pool.layers[i], s.kv_lens, s.pages, s.cu_q, s.cu_kv,
                                              s.dist, s.mask, s.sink, sliding_window=window, **s.opts)
            outs.append(o[: s.T])  # rows past the batch's tokens are padding
        return outs, s.out_cache
    if c["kind"] == "mla":
        if c["dtype"] == "bf16":
            o, _ = s.backend(s.q, s.k, s.k, s.layer, s.batch, s.pool, q_rope=s.q_rope, k_rope=s.k_rope)
        else:
            o, _ = pkg.mla_ragged_paged_attention(s.q, s.q_rope, s.k, s.k_rope, s.cache, s.kv_lens, s.pages, s.cu_q, s.cu_kv,
                                                  s.dist, sm_scale=s.scale, **s.opts)
        return o, s.out_cache
    common = dict(sm_scale=s.scale, page_size=c["page"], pages_per_seq=s.pages_per_seq, kv_lora_rank=LATENT)
    args = (s.q, s.q_rope, s.k, s.k_rope, s.cache, s.kv_lens, s.topk, s.pages, s.cu_q, s.cu_kv, s.dist)
    if c["level"] == "page":
        o, _ = pkg.sparse_mla_page_level(*args, k_pages_max=c["kp"], **common)
        return o, s.out_cache
    return pkg.sparse_mla_via_dense(*args, **common)
