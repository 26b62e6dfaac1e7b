"""GPU parity of the sparse absorbed-MLA wrappers (sglang-jax_amd/dsa.py) against the CPU oracles:
token-level selection against the restated sparse reference (dsa/ref.py:272-337), page-level
selection against the dense MLA oracle over the page lists worked out in plain loops
(dsa/sparse_mla.py:107-175).  rtol = atol = 2e-2 (bf16)."""

import ctypes
import sys

import numpy as np
import pytest
import torch

from parity import assert_parity

from oracle.ref_dsa import page_level_metadata_ref, sparse_mla_ref, topk_pages_ref
from oracle.ref_mla import ref_mla_ragged_paged_attention

pytestmark = pytest.mark.gpu
TOL = dict(rtol=2e-2, atol=2e-2)


@pytest.fixture(autouse=True)
def no_waves(request, monkeypatch):
    if getattr(request, "param", False):
        monkeypatch.setenv("RPA_MLA_WAVES", "0")


# With the kernels that the plans choose, and without those of a wave per tile.
both_ways = pytest.mark.parametrize("no_waves", [False, True], ids=["by_call", "no_waves"], indirect=True)


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def batch(wl, kv_lens, P, seed, Hq=16):
    b = wl.make_mla_batch("dsa", [1] * len(kv_lens), kv_lens, num_q_heads=Hq, lkv_dim=512, rope_dim=64, page_size=P,
                          seed=seed, sm_scale=192 ** -0.5)
    # one more page at the end: the padding target, owned by no sequence
    b.cache_kv = torch.cat([b.cache_kv, torch.zeros_like(b.cache_kv[:1])], dim=0)
    return b


def draw_topk(kv_lens, k, seed):
    """k positions per sequence, the newest token last among the valid ones, -1 padded."""
    rng = np.random.default_rng(seed)
    out = np.full((len(kv_lens), k), -1, dtype=np.int32)
    for i, n in enumerate(kv_lens):
        m = min(k, n)
        older = rng.choice(n - 1, size=m - 1, replace=False) if m > 1 else np.zeros(0, dtype=np.int64)
        out[i, : m - 1] = older
        out[i, m - 1] = n - 1
    return out


@pytest.mark.parametrize("P", [16, 64])
def test_topk_pages_on_the_device(pkg, gpu, P):
    kv_lens = [40, 300, 64, 1000, 130]
    topk = draw_topk(kv_lens, 48, 5)
    pps = -(-max(kv_lens) // P)
    for kp in (4, 64):
        got = pkg.compute_topk_pages(torch.from_numpy(topk).to(gpu), page_size=P, pages_per_seq=pps, k_pages_max=kp)
        assert np.array_equal(got.cpu().numpy(), topk_pages_ref(topk, P, pps, kp))


@both_ways
@pytest.mark.parametrize("with_new_token", [False, True])
def test_token_level_selection_through_the_dense_kernel(pkg, wl, gpu, with_new_token):
    kv_lens, P, k = [40, 300, 64, 1000, 130], 16, 64
    b = batch(wl, kv_lens, P, 81)
    topk = torch.from_numpy(draw_topk(kv_lens, k, 6))
    S = len(kv_lens)
    pps = -(-max(kv_lens) // P)
    pages = torch.cat([b.page_indices, torch.zeros(pps, dtype=torch.int32)])
    q = torch.cat([b.ql_nope, b.q_pe], dim=-1)
    say(f"dsa via dense new_token={with_new_token}")
    want = sparse_mla_ref(q, b.cache_kv, b.kv_lens, topk, pages, b.cu_q_lens, b.cu_kv_lens, [S, S, S],
                          sm_scale=b.sm_scale, pages_per_seq=pps, v_dim=512)
    g = b.to(gpu)
    cache = b.cache_kv.clone()
    new_c = new_r = None
    if with_new_token:
        # the newest row of every sequence is not in the cache yet: it arrives as new_kv_c / new_k_pe
        new_c = torch.zeros(S, 512, dtype=torch.bfloat16)
        new_r = torch.zeros(S, 64, dtype=torch.bfloat16)
        o = 0
        for i, n in enumerate(kv_lens):
            page, off = int(b.page_indices[o + (n - 1) // P]), (n - 1) % P
            new_c[i], new_r[i] = cache[page, off, :512], cache[page, off, 512:]
            cache[page, off] = float("nan")
            o += -(-n // P)
        new_c, new_r = new_c.to(gpu), new_r.to(gpu)
    got = pkg.sparse_mla_via_dense(
        g.ql_nope, g.q_pe, new_c, new_r, cache.to(gpu), g.kv_lens, topk.to(gpu), g.page_indices, g.cu_q_lens,
        g.cu_kv_lens, (S, S, S), sm_scale=b.sm_scale, page_size=P, pages_per_seq=pps, kv_lora_rank=512)
    torch.cuda.synchronize()
    assert_parity(got.cpu().float(), want.float(), **TOL)


@both_ways
@pytest.mark.parametrize("precomputed", [False, True])
def test_page_level_selection(pkg, wl, gpu, precomputed):
    kv_lens, P, k, kp = [40, 300, 64, 1000, 130], 16, 24, 32
    b = batch(wl, kv_lens, P, 82)
    topk_np = draw_topk(kv_lens, k, 7)
    S = len(kv_lens)
    pps = -(-max(kv_lens) // P)
    sentinel = b.cache_kv.shape[0] - 1
    sp_len, sp_pages = page_level_metadata_ref(b.kv_lens.numpy(), topk_np, b.page_indices.numpy(), b.cu_q_lens.numpy(),
                                               b.cu_kv_lens.numpy(), page_size=P, pages_per_seq=pps, k_pages_max=kp,
                                               sentinel_page=sentinel)
    want, _ = ref_mla_ragged_paged_attention(
        b.ql_nope, b.q_pe, None, None, b.cache_kv, torch.from_numpy(sp_len), torch.from_numpy(sp_pages).reshape(-1),
        torch.arange(S + 1, dtype=torch.int32), [S, S, S], sm_scale=b.sm_scale)
    # the newest row arrives as new_kv_c / new_k_pe and must land in its true slot
    cache = b.cache_kv.clone()
    new_c = torch.zeros(S, 512, dtype=torch.bfloat16)
    new_r = torch.zeros(S, 64, dtype=torch.bfloat16)
    o = 0
    for i, n in enumerate(kv_lens):
        page, off = int(b.page_indices[o + (n - 1) // P]), (n - 1) % P
        new_c[i], new_r[i] = cache[page, off, :512], cache[page, off, 512:]
        cache[page, off] = 0
        o += -(-n // P)
    g = b.to(gpu)
    topk = torch.from_numpy(topk_np).to(gpu)
    pre = pkg.compute_topk_pages(topk, page_size=P, pages_per_seq=pps, k_pages_max=kp) if precomputed else None
    say(f"dsa page level precomputed={precomputed}")
    got, cache_out = pkg.sparse_mla_page_level(
        g.ql_nope, g.q_pe, new_c.to(gpu), new_r.to(gpu), cache.to(gpu), g.kv_lens, topk, g.page_indices, g.cu_q_lens,
        g.cu_kv_lens, (S, S, S), pre, sm_scale=b.sm_scale, page_size=P, pages_per_seq=pps, kv_lora_rank=512,
        k_pages_max=kp)
    torch.cuda.synchronize()
    assert_parity(got.cpu().float(), want.float(), **TOL)
    assert torch.equal(cache_out.cpu(), b.cache_kv)  # every new row back in its slot, nothing else touched


@both_ways
@pytest.mark.parametrize("level", ["page", "token"])
@pytest.mark.parametrize("P,Hq,k,dtype", [(16, 16, 2048, "bf16"), (64, 64, 300, "bf16"), (16, 128, 33, "bf16"), (24, 40, 65, "bf16"),
                                          (128, 32, 512, "e4m3"), (16, 128, 96, "e4m3")])
def test_selections_of_every_shape(pkg, wl, gpu, level, P, Hq, k, dtype):
    """Head counts of every workgroup shape, pages below and above a tile, selections that end inside one, rows cut in pieces;
    lengths from one token to far more than the selection."""
    check_selections(pkg, wl, gpu, level, P, Hq, k, dtype, [1, 2, 31, P, P + 1, 700, 5003], 40)


@both_ways
@pytest.mark.parametrize("level,P,Hq,k,dtype,kv_lens,kp", [
    # sequences of 2048 pages (whose ids wait in LDS) and of more, and more of them than a wave has lanes
    ("page", 16, 16, 300, "bf16", [32768, 5, 900], 40), ("page", 16, 16, 300, "bf16", [32769, 40000, 5, 900], 40),
    ("page", 32, 64, 2048, "e4m3", [70000, 33, 3000], 70), ("page", 64, 16, 64, "bf16", list(range(1, 140)), 4),
    # pieces of more than 64 pages, and a last one that ends in its 64th
    ("page", 32, 16, 2048, "bf16", [4500 + i for i in range(150)], 130), ("page", 32, 32, 2048, "bf16", [2048] * 256, 64),
    # selections of more than one batch, unused entries between valid ones aside
    ("page", 64, 128, 2600, "bf16", [2600, 6000, 1], 64), ("token", 16, 64, 2600, "bf16", [2600, 2599, 6000, 1], 0),
    ("token", 16, 16, 40, "e4m3", list(range(1, 140)), 0),
])
def test_tables_of_every_size(pkg, wl, gpu, level, P, Hq, k, dtype, kv_lens, kp):
    check_selections(pkg, wl, gpu, level, P, Hq, k, dtype, kv_lens, kp)


def check_selections(pkg, wl, gpu, level, P, Hq, k, dtype, kv_lens, kp):
    b = batch(wl, kv_lens, P, 83, Hq=Hq)
    topk_np = draw_topk(kv_lens, k, 8)
    S, pps = len(kv_lens), -(-max(kv_lens) // P)
    pages = torch.cat([b.page_indices, torch.zeros(pps, dtype=torch.int32)])
    dt = torch.float8_e4m3fn if dtype == "e4m3" else torch.bfloat16
    stored = b.cache_kv.to(dt)
    ref_cache = stored.to(torch.bfloat16)
    say(f"dsa {level} P={P} Hq={Hq} k={k} {dtype}")
    if level == "token":
        want = sparse_mla_ref(torch.cat([b.ql_nope, b.q_pe], dim=-1), ref_cache, b.kv_lens, torch.from_numpy(topk_np), pages,
                              b.cu_q_lens, b.cu_kv_lens, [S, S, S], sm_scale=b.sm_scale, pages_per_seq=pps, v_dim=512)
    else:
        sp_len, sp_pages = page_level_metadata_ref(b.kv_lens.numpy(), topk_np, b.page_indices.numpy(), b.cu_q_lens.numpy(),
                                                   b.cu_kv_lens.numpy(), page_size=P, pages_per_seq=pps, k_pages_max=kp,
                                                   sentinel_page=stored.shape[0] - 1)
        want, _ = ref_mla_ragged_paged_attention(
            b.ql_nope, b.q_pe, None, None, ref_cache, torch.from_numpy(sp_len), torch.from_numpy(sp_pages).reshape(-1),
            torch.arange(S + 1, dtype=torch.int32), [S, S, S], sm_scale=b.sm_scale)
    new_c = torch.zeros(S, 512, dtype=torch.bfloat16).to(dt)
    new_r = torch.zeros(S, 64, dtype=torch.bfloat16).to(dt)
    cache, o = stored.clone(), 0
    for i, n in enumerate(kv_lens):
        page, off = int(b.page_indices[o + (n - 1) // P]), (n - 1) % P
        new_c[i], new_r[i] = cache[page, off, :512], cache[page, off, 512:]
        cache.view(torch.uint8)[page, off] = 0
        o += -(-n // P)
    g, cache = b.to(gpu), cache.to(gpu)
    args = (g.ql_nope, g.q_pe, new_c.to(gpu), new_r.to(gpu), cache, g.kv_lens, torch.from_numpy(topk_np).to(gpu), g.page_indices,
            g.cu_q_lens, g.cu_kv_lens, (S, S, S))
    common = dict(sm_scale=b.sm_scale, page_size=P, pages_per_seq=pps, kv_lora_rank=512)
    if level == "token":
        before = cache.view(torch.uint8).clone()
        got = pkg.sparse_mla_via_dense(*args, **common)
        assert torch.equal(cache.view(torch.uint8), before)
    else:
        got, cache_out = pkg.sparse_mla_page_level(*args, k_pages_max=kp, **common)
        assert torch.equal(cache_out.cpu().view(torch.uint8), stored.view(torch.uint8))
    torch.cuda.synchronize()
    assert_parity(got.cpu().float(), want.float(), **TOL)


class SparseParams(ctypes.Structure):  # RpaMlaSparse of include/rpa.h
    _fields_ = [("topk", ctypes.c_void_p)] + [(n, ctypes.c_int32) for n in (
        "topk_count", "topk_stride", "topk_is_pages", "pages_per_seq", "k_pages_max", "num_page_indices")]


@both_ways
@pytest.mark.parametrize("window", [1, 33, 700])
@pytest.mark.parametrize("level,P,Hq,dtype", [
    ("page", 64, 16, "bf16"), ("page", 64, 128, "bf16"), ("page", 16, 128, "bf16"), ("page", 24, 96, "bf16"), ("page", 32, 64, "e4m3"),
    ("token", 64, 32, "bf16"), ("token", 16, 128, "e4m3"),
])
def test_a_window_over_a_selection(pkg, wl, gpu, level, P, Hq, dtype, window):
    """The C entry takes the batch as rpa_mla_decode does, its window too: the last `window` tokens of a selection, in rows that stay
    whole and in rows cut into pieces."""
    kv_lens, k, kp = [1, 31, P + 1, 900, 5003], 2048, 40
    b = batch(wl, kv_lens, P, 84, Hq=Hq)
    S, pps = len(kv_lens), -(-max(kv_lens) // P)
    topk_np = draw_topk(kv_lens, k, 9)
    stored = b.cache_kv.to(torch.float8_e4m3fn if dtype == "e4m3" else torch.bfloat16)
    say(f"dsa window {level} P={P} Hq={Hq} {dtype} window={window}")
    if level == "token":
        seen = np.full_like(topk_np, -1)
        for i, n in enumerate(kv_lens):
            valid = topk_np[i, : min(k, n)][-window:]
            seen[i, : len(valid)] = valid
        pages = torch.cat([b.page_indices, torch.zeros(pps, dtype=torch.int32)])
        want = sparse_mla_ref(torch.cat([b.ql_nope, b.q_pe], dim=-1), stored.to(torch.bfloat16), b.kv_lens, torch.from_numpy(seen), pages,
                              b.cu_q_lens, b.cu_kv_lens, [S, S, S], sm_scale=b.sm_scale, pages_per_seq=pps, v_dim=512)
    else:
        sp_len, sp_pages = page_level_metadata_ref(b.kv_lens.numpy(), topk_np, b.page_indices.numpy(), b.cu_q_lens.numpy(),
                                                   b.cu_kv_lens.numpy(), page_size=P, pages_per_seq=pps, k_pages_max=kp,
                                                   sentinel_page=stored.shape[0] - 1)
        want, _ = ref_mla_ragged_paged_attention(
            b.ql_nope, b.q_pe, None, None, stored.to(torch.bfloat16), torch.from_numpy(sp_len), torch.from_numpy(sp_pages).reshape(-1),
            torch.arange(S + 1, dtype=torch.int32), [S, S, S], sm_scale=b.sm_scale, sliding_window=window)
    g, cache, topk = b.to(gpu), stored.to(gpu), torch.from_numpy(topk_np).to(gpu)
    out = torch.full_like(g.ql_nope, float("nan"))
    p = pkg._lib.RpaMlaParams(
        ql_nope=g.ql_nope.data_ptr(), q_pe=g.q_pe.data_ptr(), out=out.data_ptr(), cache_kv=cache.data_ptr(), kv_lens=g.kv_lens.data_ptr(),
        page_indices=g.page_indices.data_ptr(), cu_q_lens=g.cu_q_lens.data_ptr(), cu_kv_lens=g.cu_kv_lens.data_ptr(), num_tokens=S,
        num_seqs=S, num_q_heads=Hq, lkv_dim=512, rope_dim=64, row_stride=cache.shape[-1], rope_offset=512, page_size=P,
        total_pages=cache.shape[0], sliding_window=window, sm_scale=b.sm_scale,
        cache_dtype=pkg._lib.RPA_KV_FP8_E4M3 if dtype == "e4m3" else pkg._lib.RPA_KV_BF16)
    s = SparseParams(topk=topk.data_ptr(), topk_count=k, topk_stride=k, pages_per_seq=pps, k_pages_max=kp if level == "page" else 0,
                     num_page_indices=g.page_indices.numel())
    lib = pkg._lib.load()
    size, run = lib.rpa_mla_sparse_workspace_bytes, lib.rpa_mla_sparse_attention
    size.restype, size.argtypes = ctypes.c_size_t, [ctypes.c_void_p] * 2
    run.restype, run.argtypes = ctypes.c_int, [ctypes.c_void_p] * 5
    ws = torch.full((size(ctypes.byref(p), ctypes.byref(s)),), 0xFF, dtype=torch.uint8, device=gpu)
    p.workspace, p.workspace_bytes = ws.data_ptr(), ws.numel()
    assert run(ctypes.byref(p), ctypes.byref(s), None, None, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert_parity(out.cpu().float(), want.float(), **TOL)


@pytest.mark.parametrize("level,P,Hq,dtype", [("page", 64, 16, "bf16"), ("page", 24, 40, "e4m3"), ("token", 64, 16, "bf16"), ("token", 16, 128, "e4m3")])
def test_selections_with_new_rows_anywhere_in_memory(pkg, wl, gpu, monkeypatch, level, P, Hq, dtype):
    """New rows that begin 8 bytes behind a multiple of 16 go through registers on a wave per tile as well: the same output and cache, bit for bit."""
    monkeypatch.setenv("RPA_MLA_WAVES", "1")
    kv_lens, k = [1, 63, 64, 65, 700, 3001], 512
    b = batch(wl, kv_lens, P, 86, Hq=Hq)
    S, pps, dt = len(kv_lens), -(-max(kv_lens) // P), torch.float8_e4m3fn if dtype == "e4m3" else torch.bfloat16
    g, stored, topk = b.to(gpu), b.cache_kv.to(dt).to(gpu), torch.from_numpy(draw_topk(kv_lens, k, 10)).to(gpu)
    n, rows, got = 16 // dt.itemsize // 2, torch.randn(S, 576, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16).to(dt).to(gpu), []
    for off in (0, n):
        parts = []
        for part in (rows[:, :512], rows[:, 512:]):
            room = torch.zeros(part.numel() + n, dtype=dt, device=gpu)
            room[off:off + part.numel()] = part.reshape(-1)
            parts.append(room[off:off + part.numel()].view(part.shape))
            assert parts[-1].data_ptr() % 16 == (8 if off else 0)
        cache = stored.clone()
        say(f"dsa {level} new rows at +{off} P={P} Hq={Hq} {dtype}")
        args = (g.ql_nope, g.q_pe, *parts, cache, g.kv_lens, topk, g.page_indices, g.cu_q_lens, g.cu_kv_lens, (S, S, S))
        common = dict(sm_scale=b.sm_scale, page_size=P, pages_per_seq=pps, kv_lora_rank=512)
        out = pkg.sparse_mla_via_dense(*args, **common) if level == "token" else pkg.sparse_mla_page_level(*args, k_pages_max=40, **common)[0]
        torch.cuda.synchronize()
        got.append((out, cache.view(torch.uint8)))
    assert torch.isfinite(got[0][0]).all() and torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("level,P,dtype,S,waves", [("page", 64, "bf16", 15, "0"), ("page", 64, "bf16", 16, "1"), ("page", 64, "e4m3", 3, "0"), ("page", 64, "e4m3", 4, "1"), ("page", 16, "bf16", 3, "1"),
                                                   ("token", 64, "bf16", 3, "1")])
def test_few_selections_of_whole_pages_share_tiles(pkg, wl, gpu, monkeypatch, level, P, dtype, S, waves):
    """16 heads, pages of whole tiles: under four rounds of 64 tokens per CU (e4m3: one) the waves of a workgroup share its tiles, from there on, and for
    every other selection, each has its own.  Which one ran shows in the bits, and both are near the oracle."""
    kv_lens, k = [4100] + [100 + 37 * i for i in range(S - 1)], 256
    b = batch(wl, kv_lens, P, 87)
    pps, dt = -(-max(kv_lens) // P), torch.float8_e4m3fn if dtype == "e4m3" else torch.bfloat16
    g, cache, topk_np, got = b.to(gpu), b.cache_kv.to(dt).to(gpu), draw_topk(kv_lens, k, 11), {}
    args = (g.ql_nope, g.q_pe, None, None, cache, g.kv_lens, torch.from_numpy(topk_np).to(gpu), g.page_indices, g.cu_q_lens, g.cu_kv_lens, (S, S, S))
    common = dict(sm_scale=b.sm_scale, page_size=P, pages_per_seq=pps, kv_lora_rank=512)
    for way in (None, "0", "1"):
        monkeypatch.setenv("RPA_MLA_WAVES", way) if way else monkeypatch.delenv("RPA_MLA_WAVES", raising=False)
        say(f"dsa {level} P={P} {dtype} S={S} RPA_MLA_WAVES={way}")
        out = pkg.sparse_mla_via_dense(*args, **common) if level == "token" else pkg.sparse_mla_page_level(*args, k_pages_max=64, **common)[0]
        torch.cuda.synchronize()
        got[way] = out.cpu()
    assert torch.equal(got[None], got[waves]) and not torch.equal(got["0"], got["1"])
    assert_parity(got["0"].float(), got["1"].float(), **TOL)
