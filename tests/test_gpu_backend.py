"""The attention backend end to end on the GPU: metadata from a scheduler-shaped batch,
per-layer calls that write the new tokens into the layer's cache and attend over it
(flashattention_backend.py:146-237, 603-760), checked against the CPU oracle run on the
complete cache."""

import sys
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from parity import assert_parity

from oracle.ref_rpa import ref_ragged_paged_attention_fused

pytestmark = pytest.mark.gpu

TOL = dict(rtol=2e-2, atol=2e-2)


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


class Pool:
    """Per-layer fused caches [pages, P, 2*Hkv, D] (memory_pool.py:566-611)."""

    def __init__(self, layers, pages, P, Hkv, D, device, seed):
        g = torch.Generator().manual_seed(seed)
        # unused slots hold NaN canaries: nothing may read them
        self.host = [torch.full((pages, P, 2 * Hkv, D), float("nan"), dtype=torch.bfloat16) for _ in range(layers)]
        self.dev = [h.to(device) for h in self.host]
        self.g = g

    def get_fused_kv_buffer(self, layer_id):
        return self.dev[layer_id]


def padded_table(page_lists, width):
    t = np.zeros((len(page_lists), width), dtype=np.int32)
    for i, ps in enumerate(page_lists):
        t[i, :len(ps)] = ps
    return torch.from_numpy(t)


@pytest.mark.parametrize("P,window,cap", [(16, None, None), (64, 48, 30.0)])
def test_extend_then_decode_steps(pkg, gpu, P, window, cap):
    Hq, Hkv, D, layers, pool_pages = 8, 2, 128, 2, 96
    rng = np.random.default_rng(7)
    gen = torch.Generator().manual_seed(11)
    pool = Pool(layers, pool_pages, P, Hkv, D, gpu, 3)
    backend = pkg.FlashAttention(Hq, Hkv, D, page_size=P, device=gpu)
    layer_objs = [SimpleNamespace(layer_id=i, scaling=D ** -0.5, head_dim=D, sliding_window_size=window,
                                  logit_cap=cap, xai_temperature_len=-1, softmax_dtype=None, attn_type=None)
                  for i in range(layers)]
    free = list(rng.permutation(pool_pages))
    prompt = [37, 70, 5]
    bs_pad = 4  # one padded (empty) request slot, as the scheduler's bucketing leaves them
    pages = [[] for _ in range(bs_pad)]
    seq_lens = np.zeros(bs_pad, dtype=np.int32)
    # what each layer's cache holds per sequence (host truth), for the oracle
    truth = [[torch.zeros(0, 2 * Hkv, D, dtype=torch.bfloat16) for _ in range(bs_pad)] for _ in range(layers)]

    def run_step(mode, new_lens):
        nonlocal seq_lens
        new_lens = np.asarray(new_lens, dtype=np.int32)
        seq_lens = seq_lens + new_lens
        for i in range(bs_pad):
            while len(pages[i]) * P < seq_lens[i]:
                pages[i].append(int(free.pop()))
        cache_loc = np.concatenate([np.arange(p * P, p * P + P) for ps in pages for p in ps]).astype(np.int32)
        batch = SimpleNamespace(forward_mode=mode, seq_lens=seq_lens.copy(), cache_loc=cache_loc,
                                extend_seq_lens=new_lens, dp_size=1, per_dp_bs_size=bs_pad)
        backend.forward_metadata = backend.get_forward_metadata(batch)
        T = int(new_lens.sum())
        n_real = int((seq_lens > 0).sum())
        for L in range(layers):
            q = torch.randn(T, Hq * D, generator=gen).to(torch.bfloat16)
            k = torch.randn(T, Hkv * D, generator=gen).to(torch.bfloat16)
            v = torch.randn(T, Hkv * D, generator=gen).to(torch.bfloat16)
            out, cache = backend(q.to(gpu), k.to(gpu), v.to(gpu), layer_objs[L], batch, pool)
            torch.cuda.synchronize()
            assert out.shape == (T, Hq * D)
            assert cache.data_ptr() == pool.dev[L].data_ptr()
            # host truth: append the new tokens (K0,V0,K1,V1,... head order)
            t = 0
            for i in range(bs_pad):
                for _ in range(int(new_lens[i])):
                    row = torch.stack([k[t].view(Hkv, D), v[t].view(Hkv, D)], dim=1).reshape(1, 2 * Hkv, D)
                    truth[L][i] = torch.cat([truth[L][i], row])
                    t += 1
            full = torch.zeros(pool_pages, P, 2 * Hkv, D, dtype=torch.bfloat16)
            for i in range(bs_pad):
                for j, pg in enumerate(pages[i]):
                    rows = truth[L][i][j * P:(j + 1) * P]
                    full[pg, :len(rows)] = rows
            cu_q = np.concatenate([[0], np.cumsum(new_lens)]).astype(np.int32)
            want = ref_ragged_paged_attention_fused(
                q.view(T, Hq, D), full, torch.from_numpy(seq_lens.copy()), padded_table(pages, 8),
                torch.from_numpy(cu_q), [n_real], sm_scale=D ** -0.5, sliding_window=window, soft_cap=cap)
            assert_parity(out.cpu().float().view(T, Hq, D), want.float(), **TOL)
            # every written slot equals the host truth bit for bit; the rest is untouched (NaN)
            got_cache = pool.dev[L].cpu()
            for i in range(bs_pad):
                for j, pg in enumerate(pages[i]):
                    rows = truth[L][i][j * P:(j + 1) * P]
                    assert torch.equal(got_cache[pg, :len(rows)].view(torch.int16), rows.view(torch.int16))
                    assert torch.isnan(got_cache[pg, len(rows):].float()).all()

    say(f"extend P={P} window={window} cap={cap}")
    run_step(pkg.ForwardMode.EXTEND, prompt + [0])
    assert backend.forward_metadata.host_distribution.tolist() == [0, 3, 3]
    for step in range(3):
        say(f"decode step {step}")
        run_step(pkg.ForwardMode.DECODE, [1, 1, 1, 0])
        assert backend.forward_metadata.host_distribution.tolist() == [3, 3, 3]
    say("chunked extend on top of the existing prefix")
    run_step(pkg.ForwardMode.EXTEND, [9, 4, 33, 0])


def test_mla_backend_extend_then_decode(pkg, gpu):
    """MLAAttentionBackend (mla_backend.py:83-389): prompt, then decode steps, on the
    reference's 640-wide latent rows; output and cache against the CPU oracle."""
    from oracle.ref_mla import ref_mla_ragged_paged_attention

    Hq, P, pool_pages, W = 16, 16, 48, 640
    rng = np.random.default_rng(17)
    gen = torch.Generator().manual_seed(19)
    host_cache = torch.zeros(pool_pages, P, W, dtype=torch.bfloat16)
    pool = SimpleNamespace(buf=host_cache.to(gpu))
    pool.get_fused_kv_buffer = lambda layer_id: pool.buf
    backend = pkg.MLAAttentionBackend(Hq, 512, 128, 64, 128, page_size=P, device=gpu)
    layer = SimpleNamespace(layer_id=0, scaling=None, sliding_window_size=None, logit_cap=None)
    free = list(rng.permutation(pool_pages))
    bs = 3
    pages = [[] for _ in range(bs)]
    seq_lens = np.zeros(bs, dtype=np.int32)

    def step(mode, new_lens):
        nonlocal seq_lens, host_cache
        new_lens = np.asarray(new_lens, dtype=np.int32)
        seq_lens = seq_lens + new_lens
        for i in range(bs):
            while len(pages[i]) * P < seq_lens[i]:
                pages[i].append(int(free.pop()))
        cache_loc = np.concatenate([np.arange(p * P, p * P + P) for ps in pages for p in ps]).astype(np.int32)
        batch = SimpleNamespace(forward_mode=mode, seq_lens=seq_lens.copy(), cache_loc=cache_loc,
                                extend_seq_lens=new_lens, dp_size=1, per_dp_bs_size=bs)
        backend.forward_metadata = backend.get_forward_metadata(batch)
        T = int(new_lens.sum())
        q = (torch.randn(T, Hq, 512, generator=gen) * 0.5).to(torch.bfloat16)
        qr = (torch.randn(T, Hq, 64, generator=gen) * 0.5).to(torch.bfloat16)
        kc = (torch.randn(T, 1, 512, generator=gen) * 0.5).to(torch.bfloat16)
        kr = (torch.randn(T, 1, 64, generator=gen) * 0.5).to(torch.bfloat16)
        out, cache = backend(q.to(gpu), kc.to(gpu), kc.to(gpu), layer, batch, pool, q_rope=qr.to(gpu), k_rope=kr.to(gpu))
        torch.cuda.synchronize()
        width = max(len(p) for p in pages)
        table = np.zeros((bs, width), dtype=np.int32)
        for i, ps in enumerate(pages):
            table[i, :len(ps)] = ps
        cu_q = np.concatenate([[0], np.cumsum(new_lens)]).astype(np.int32)
        want, host_cache = ref_mla_ragged_paged_attention(
            q, qr, kc[:, 0], kr[:, 0], host_cache, torch.from_numpy(seq_lens.copy()),
            torch.from_numpy(table.reshape(-1)), torch.from_numpy(cu_q), [0, 0, bs],
            sm_scale=1.0 / np.sqrt(192.0), layout="padded")
        assert torch.equal(cache.cpu().view(torch.int16), host_cache.view(torch.int16))
        assert_parity(out.cpu().float(), want.float(), **TOL)

    say("mla extend")
    step(pkg.ForwardMode.EXTEND, [37, 70, 5])
    assert backend.forward_metadata.host_distribution.tolist() == [0, 0, 3]
    for s_ in range(2):
        say(f"mla decode {s_}")
        step(pkg.ForwardMode.DECODE, [1, 1, 1])


@pytest.mark.parametrize("P,lens", [(16, [1]), (16, [17, 0, 5]), (1, [300, 800, 500]), (16, [9000, 40000, 7, 0])])
@pytest.mark.parametrize("mixed", [False, True])
def test_metadata_in_one_upload(pkg, gpu, P, lens, mixed):
    """The native metadata against the numpy builder, from one launch's worth of words to more than kernel arguments carry."""
    rng = np.random.default_rng(5)
    kv = np.array(lens, dtype=np.int32)
    pages = rng.permutation(int((-(-kv // P)).sum()) + 3).astype(np.int32)
    loc = (pages[: int((-(-kv // P)).sum())].astype(np.int64)[:, None] * P + np.arange(P)).reshape(-1).astype(np.int32)
    for mode, ext in ((pkg.ForwardMode.DECODE, None), (pkg.ForwardMode.EXTEND, np.minimum(kv, 5))):
        batch = SimpleNamespace(forward_mode=mode, seq_lens=kv, cache_loc=loc, extend_seq_lens=ext, dp_size=1, per_dp_bs_size=len(kv))
        backend = (pkg.MLAAttentionBackend(16, 512, 128, 64, 128, page_size=P, device=gpu) if mixed and P > 1
                   else pkg.FlashAttention(8, 2, 128, page_size=P, device=gpu))
        md = backend.get_forward_metadata(batch)
        want = pkg.build_forward_metadata(forward_mode=mode, seq_lens=kv, cache_loc=loc, extend_seq_lens=ext, page_size=P,
                                          extend_distribution_is_mixed=isinstance(backend, pkg.MLAAttentionBackend))
        for name in ("cu_q_lens", "cu_kv_lens", "page_indices", "seq_lens", "distribution"):
            got = getattr(md, name)
            assert got.dtype == torch.int32 and np.array_equal(got.cpu().numpy(), want[name]), name
        assert np.array_equal(md.host_distribution, want["distribution"])
        assert md.max_kv_len == kv.max() and md.max_q_len == (1 if ext is None else ext.max())


@pytest.mark.parametrize("P,D,Hq,Hkv,dtype,window,cap", [
    (64, 128, 8, 2, torch.bfloat16, None, None), (16, 128, 16, 4, torch.bfloat16, 100, None), (1, 128, 8, 4, torch.bfloat16, None, 30.0),
    (24, 256, 8, 2, torch.bfloat16, None, None), (16, 128, 8, 1, torch.float8_e4m3fn, None, None),
    (64, 256, 4, 2, torch.float8_e4m3fn, 64, 50.0)])
@pytest.mark.parametrize("lens", [[1003], [130, 1, 70, 300, 64], [2500, 129]])
def test_prompts_attend_to_the_rows_they_bring(pkg, gpu, P, D, Hq, Hkv, dtype, window, cap, lens):
    """Prompts without a prefix read the caller's keys and values and fill the cache beside the attention; the functional
    operator on the same batch writes first and reads the cache.  Both against 64 bits."""
    gen = torch.Generator().manual_seed(3)
    rng = np.random.default_rng(4)
    kv = np.array(lens, dtype=np.int32)
    n = int((-(-kv // P)).sum())
    pages = rng.permutation(n + 2)[:n].astype(np.int32)
    loc = (pages.astype(np.int64)[:, None] * P + np.arange(P)).reshape(-1).astype(np.int32)
    T = int(kv.sum())
    cache = torch.full((n + 2, P, 2 * Hkv, D), 3.0).to(dtype).to(gpu)
    other = cache.clone()
    q = torch.randn(T, Hq, D, generator=gen).to(torch.bfloat16).to(gpu)
    k, v = (torch.randn(T, Hkv, D, generator=gen).to(dtype).to(gpu) for _ in range(2))
    backend = pkg.FlashAttention(Hq, Hkv, D, page_size=P, device=gpu)
    batch = SimpleNamespace(forward_mode=pkg.ForwardMode.EXTEND, seq_lens=kv, cache_loc=loc, extend_seq_lens=kv, dp_size=1,
                            per_dp_bs_size=len(kv))
    md = backend.forward_metadata = backend.get_forward_metadata(batch)
    assert md.no_prefix
    layer = SimpleNamespace(layer_id=0, scaling=D ** -0.5, head_dim=D, sliding_window_size=window, logit_cap=cap)
    say(f"prompts P={P} D={D} {dtype} window={window} cap={cap} {lens}")
    out, _ = backend(q.view(T, -1), k.view(T, -1), v.view(T, -1), layer, batch, SimpleNamespace(get_fused_kv_buffer=lambda i: cache))
    want, _ = pkg.ragged_paged_attention(q, k, v, other, md.seq_lens, md.page_indices, md.cu_q_lens, md.cu_kv_lens, md.host_distribution,
                                         sm_scale=D ** -0.5, sliding_window=window, soft_cap=cap, max_kv_len=md.max_kv_len,
                                         max_q_len=md.max_q_len)
    torch.cuda.synchronize()
    assert torch.equal(cache.view(torch.uint8), other.view(torch.uint8))
    assert_parity(out.view(T, Hq, D).cpu().float(), want.cpu().float(), **TOL)
    exact = attention64(q, k, v, lens, D ** -0.5, window, cap)
    assert_parity(out.view(T, Hq, D), exact, **TOL)
    assert_parity(want, exact, **TOL)


def attention64(q, k, v, lens, scale, window=None, cap=None):
    """Prompts without a prefix in 64 bits: [T, Hq, D] of q [T, Hq, D], k / v [T, Hkv, D]."""
    q, k, v = (x.cpu().float().double() for x in (q, k, v))
    g = q.shape[1] // k.shape[1]
    out, at = [], 0
    for n in lens:
        s = slice(at, at + n)
        at += n
        kk, vv = (x[s].repeat_interleave(g, dim=1).transpose(0, 1) for x in (k, v))
        x = q[s].transpose(0, 1) @ kk.transpose(1, 2) * scale
        x = cap * torch.tanh(x / cap) if cap else x
        row, col = torch.arange(n)[:, None], torch.arange(n)[None, :]
        x = x.masked_fill((col > row) | (col <= row - (window or n + 1)), -torch.inf)
        out.append((torch.softmax(x, dim=-1) @ vv).transpose(0, 1))
    return torch.cat(out)


# The 2-norm of the whole error over that of the result.  Scores scaled in 32 bits: probabilities and results rounded to
# bf16 once (each up to 2^-8 of the value, 2^-8 / sqrt(12) / ~0.72 = 1.6e-3 on average over the mantissas): 2.2e-3 together
# where few keys carry a row, less where many do.  Queries rounded to bf16 a second time (pages of 2^k >= 64 tokens: the
# assembly kernel) move every logit by 1.6e-3 of its own terms, 2 units of spread here: 3.2e-3 more.
@pytest.mark.parametrize("P,bound", [(1, 2.4e-3), (16, 2.4e-3), (24, 2.4e-3), (96, 2.4e-3), (64, 4.4e-3)])
@pytest.mark.parametrize("lens", [[1003], [130, 1, 70, 300, 64]])
def test_prompts_keep_the_precision_of_their_pages(pkg, gpu, P, bound, lens):
    """What reads the caller's rows suits any pages, but a kernel that rounds more is not chosen for that: prompts on pages
    that the assembly kernel does not take scale their scores in 32 bits, as the cache's rows do.  Against 64 bits, logits
    of a few units, through the layer call and through the operator that reads the cache."""
    gen = torch.Generator().manual_seed(11)
    Hq, Hkv, D = 8, 2, 128
    kv = np.array(lens, dtype=np.int32)
    n = int((-(-kv // P)).sum())
    pages = np.random.default_rng(4).permutation(n + 2)[:n].astype(np.int32)
    loc = (pages.astype(np.int64)[:, None] * P + np.arange(P)).reshape(-1).astype(np.int32)
    T = int(kv.sum())
    cache = torch.zeros(n + 2, P, 2 * Hkv, D, dtype=torch.bfloat16, device=gpu)
    q = (2 * torch.randn(T, Hq, D, generator=gen)).to(torch.bfloat16).to(gpu)
    k, v = (torch.randn(T, Hkv, D, generator=gen).to(torch.bfloat16).to(gpu) for _ in range(2))
    backend = pkg.FlashAttention(Hq, Hkv, D, page_size=P, device=gpu)
    batch = SimpleNamespace(forward_mode=pkg.ForwardMode.EXTEND, seq_lens=kv, cache_loc=loc, extend_seq_lens=kv, dp_size=1,
                            per_dp_bs_size=len(kv))
    md = backend.forward_metadata = backend.get_forward_metadata(batch)
    layer = SimpleNamespace(layer_id=0, scaling=D ** -0.5, head_dim=D, sliding_window_size=None, logit_cap=None)
    say(f"prompt precision P={P} {lens}")
    out, _ = backend(q.view(T, -1), k.view(T, -1), v.view(T, -1), layer, batch, SimpleNamespace(get_fused_kv_buffer=lambda i: cache))
    old, _ = pkg.ragged_paged_attention(q, None, None, cache, md.seq_lens, md.page_indices, md.cu_q_lens, md.cu_kv_lens,
                                        md.host_distribution, sm_scale=D ** -0.5, max_kv_len=md.max_kv_len, max_q_len=md.max_q_len)
    want = attention64(q, k, v, lens, D ** -0.5)
    for name, got in (("layer", out.view(T, Hq, D)), ("cache", old)):
        err = float((got.cpu().double() - want).norm() / want.norm())
        say(f"  {name} {err:.3e}")
        assert err <= bound, (name, err)


@pytest.mark.parametrize("mla", [False, True])
def test_metadata_arrives_in_the_order_of_its_stream(pkg, gpu, mla):
    """Metadata built on one stream, behind work that is still running there, and read on another that waits for the first
    (the host does not wait, so without that the words need not be there)."""
    P, rng = 16, np.random.default_rng(6 + mla)
    kv = np.array([700, 33, 1500, 1], dtype=np.int32)
    n = int((-(-kv // P)).sum())
    pages = rng.permutation(n).astype(np.int32) + 1
    loc = (pages.astype(np.int64)[:, None] * P + np.arange(P)).reshape(-1).astype(np.int32)
    batch = SimpleNamespace(forward_mode=pkg.ForwardMode.DECODE, seq_lens=kv, cache_loc=loc, extend_seq_lens=None, dp_size=1,
                            per_dp_bs_size=len(kv))
    backend = (pkg.MLAAttentionBackend(16, 512, 128, 64, 128, page_size=P, device=gpu) if mla
               else pkg.FlashAttention(8, 2, 128, page_size=P, device=gpu))
    one, two = torch.cuda.Stream(gpu), torch.cuda.Stream(gpu)
    torch.cuda.synchronize()
    say(f"metadata on two streams mla={mla}")
    with torch.cuda.stream(one):
        torch.cuda._sleep(50_000_000)  # some 20 ms
        md = backend.get_forward_metadata(batch)
    two.wait_stream(one)
    with torch.cuda.stream(two):
        got = {name: getattr(md, name).cpu().numpy() for name in ("page_indices", "seq_lens", "cu_q_lens", "cu_kv_lens", "distribution")}
    torch.cuda.synchronize()
    want = pkg.build_forward_metadata(forward_mode=pkg.ForwardMode.DECODE, seq_lens=kv, cache_loc=loc, page_size=P)
    for name, x in got.items():
        assert np.array_equal(x, want[name]), name


@pytest.mark.parametrize("P,lens", [(16, [40, 7, 100]), (1, [4000, 1, 2500])])
def test_metadata_inside_a_captured_graph(pkg, gpu, P, lens):
    """Under capture the upload becomes part of the graph, words and all (also more of them than an eager call sends as kernel
    arguments); every replay leaves the same ones."""
    kv = np.array(lens, dtype=np.int32)
    n = int((-(-kv // P)).sum())
    loc = (np.arange(n, dtype=np.int64)[::-1, None] * P + np.arange(P)).reshape(-1).astype(np.int32)
    batch = SimpleNamespace(forward_mode=pkg.ForwardMode.DECODE, seq_lens=kv, cache_loc=loc, extend_seq_lens=None, dp_size=1,
                            per_dp_bs_size=len(kv))
    backend = pkg.FlashAttention(8, 2, 128, page_size=P, device=gpu)
    want = pkg.build_forward_metadata(forward_mode=pkg.ForwardMode.DECODE, seq_lens=kv, cache_loc=loc, page_size=P)
    backend.get_forward_metadata(batch)
    torch.cuda.synchronize()
    say(f"metadata under capture P={P}")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        md = backend.get_forward_metadata(batch)
    for _ in range(3):
        md.page_indices.zero_()
        backend.get_forward_metadata(batch)  # (eager work between the replays)
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(md.page_indices.cpu().numpy(), want["page_indices"])
        assert np.array_equal(md.cu_kv_lens.cpu().numpy(), want["cu_kv_lens"])


def test_threads_share_a_stream_and_its_workspace(pkg, gpu):
    """Layer calls of two threads on one stream: the launches of a call (partial rows, then their merge) stay together on the
    workspace that they share, and a call keeps the buffer it was given while the other one's grows it."""
    import threading

    Hq, Hkv, D, P = 8, 2, 128, 64
    stream = torch.cuda.Stream(gpu)

    def prepare(seed, lens):
        gen = torch.Generator().manual_seed(seed)
        kv = np.array(lens, dtype=np.int32)
        n = int((-(-kv // P)).sum())
        pages = np.random.default_rng(seed).permutation(n).astype(np.int32)
        loc = (pages.astype(np.int64)[:, None] * P + np.arange(P)).reshape(-1).astype(np.int32)
        cache = torch.randn(n, P, 2 * Hkv, D, generator=gen).to(torch.bfloat16).to(gpu)
        q, k, v = (torch.randn(len(lens), h * D, generator=gen).to(torch.bfloat16).to(gpu) for h in (Hq, Hkv, Hkv))
        backend = pkg.FlashAttention(Hq, Hkv, D, page_size=P, device=gpu)
        batch = SimpleNamespace(forward_mode=pkg.ForwardMode.DECODE, seq_lens=kv, cache_loc=loc, extend_seq_lens=None, dp_size=1,
                                per_dp_bs_size=len(lens))
        backend.forward_metadata = backend.get_forward_metadata(batch)
        layer = SimpleNamespace(layer_id=0, scaling=D ** -0.5, head_dim=D, sliding_window_size=None, logit_cap=None)
        pool = SimpleNamespace(get_fused_kv_buffer=lambda i: cache)
        return lambda: backend(q, k, v, layer, batch, pool)[0]

    rng = np.random.default_rng(2)
    calls = [prepare(1, [3000, 4100]), prepare(2, [int(x) for x in rng.integers(600, 6000, size=90)])]
    torch.cuda.synchronize()
    want = [c() for c in calls]
    torch.cuda.synchronize()
    got = [[], []]

    def work(i):
        with torch.cuda.stream(stream):
            for _ in range(150):
                got[i].append(calls[i]())

    say("two threads on one stream")
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i in range(2):
        assert len(got[i]) == 150 and all(torch.equal(x, want[i]) for x in got[i])


FORMS = {
    "plain": {}, "host_metadata": {}, "strided_new_tokens": {}, "narrow_cache_rows": {}, "f32_queries": {}, "cache_only": {},
    "distribution_on_the_device": {}, "distribution_as_a_tuple": {}, "sink_per_head": {}, "scalar_sink": {},
    "per_head_scales": {}, "scalar_scales": dict(k_scale=0.5, v_scale=2.0), "window": dict(sliding_window=np.int64(40)),
    "cap": dict(soft_cap=20), "bf16_logits": dict(softmax_dtype=torch.bfloat16), "no_mask": dict(causal=0), "bool_mask": {},
    "int_mask": {}, "bounds": dict(max_kv_len=np.int32(900), max_q_len=200, num_splits=3),
    # refused, with the same words
    "zero_window": dict(sliding_window=0), "zero_cap": dict(soft_cap=0.0), "positive_mask_value": dict(mask_value=1.0),
    "f64_softmax": dict(softmax_dtype=torch.float64), "wrong_scales": {}, "wide_metadata": {}, "chunk_of_nothing": dict(chunk_prefill_size=0)}


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.bfloat16), (256, torch.float8_e4m3fn)])
def test_native_calls_equal_the_general_ones(pkg, gpu, monkeypatch, form, D, dtype):
    """The native reader of a call's arguments against the general Python code, over the forms that it takes or leaves to it:
    the same rows and cache, or the same refusal."""
    P, Hq, Hkv, lens, new = 16, 8, 2, [700, 31, 400, 260], [1, 1, 130, 200]
    kv, cu = np.array(lens, dtype=np.int32), np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
    counts, T = -(-kv // P), sum(new)
    n = int(counts.sum())
    gen = torch.Generator().manual_seed(9)
    rnd = lambda *s: torch.randn(*s, generator=gen)  # noqa: E731
    rows = -(-D // 128) * 128 if form != "narrow_cache_rows" else D
    cache = torch.zeros(n, P, 2 * Hkv, rows)
    cache[..., :D] = rnd(n, P, 2 * Hkv, D)
    cache = cache.to(dtype).to(gpu)
    q = rnd(T, Hq, D).to(torch.float32 if form == "f32_queries" else torch.bfloat16).to(gpu)
    kv_new = rnd(T, 2 * Hkv, D).to(dtype).to(gpu)
    k, v = kv_new[:, :Hkv], kv_new[:, Hkv:]
    if form != "strided_new_tokens":
        k, v = k.contiguous(), v.contiguous()
    if form == "cache_only":
        k = v = None
    meta = [kv, np.random.default_rng(1).permutation(n).astype(np.int32), cu, np.concatenate([[0], np.cumsum(counts * P)]).astype(np.int32)]
    if form == "wide_metadata":
        meta[0] = kv.astype(np.int64)
    if form != "host_metadata":
        meta = [torch.from_numpy(x).to(gpu) for x in meta]
    dist = np.array([2, 2, 4], dtype=np.int32)
    dist = {"distribution_on_the_device": torch.from_numpy(dist).to(gpu), "distribution_as_a_tuple": (2, 2, 4)}.get(form, dist)
    mask = (torch.rand(int((np.array(new) * kv).sum()), generator=gen) < 0.7).to(gpu) if form.endswith("_mask") and form != "no_mask" else None
    sink = {"sink_per_head": rnd(Hq).to(gpu), "scalar_sink": 0.5}.get(form)
    kw = dict(sm_scale=D ** -0.5, **FORMS[form])
    if mask is not None:
        kw["causal"] = 0
        mask = mask.to(torch.int32) if form == "int_mask" else mask
    if form in ("per_head_scales", "wrong_scales"):
        kw.update(k_scale=(torch.rand(Hkv + (form == "wrong_scales"), generator=gen) + 0.5).to(gpu), v_scale=(torch.rand(Hkv, generator=gen) + 0.5).to(gpu))
    native = pkg._lib.load_torch()
    general = SimpleNamespace(attention=lambda *a: None, workspace=native.workspace)
    say(f"forms {form} D={D} {dtype}")
    results = []
    for module in (native, general):
        monkeypatch.setattr(pkg._lib, "_torch", module)
        own = cache.clone()
        try:
            out, _ = pkg.ragged_paged_attention(q, k, v, own, *meta, dist, mask, sink, **kw)
            torch.cuda.synchronize()
            results.append((out.cpu(), own.view(torch.uint8).cpu()))
        except (ValueError, NotImplementedError) as e:
            results.append((type(e), str(e)))
    (a, b), (c, d) = results
    if isinstance(b, str) or isinstance(d, str):
        assert (a, b) == (c, d)
        return
    assert torch.equal(b, d) and a.dtype == c.dtype
    assert_parity(a.float(), c.float(), **TOL)
