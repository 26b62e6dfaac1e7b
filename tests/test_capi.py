"""Host-side checks that need no GPU: the library loads, exports every symbol
include/rpa.h declares, and its validation mirrors the reference's
static/dynamic_validate_inputs
(python/sgl_jax/srt/kernels/ragged_paged_attention/ragged_paged_attention_v3.py:1314-1487)."""

import ctypes
import os
import re
import sys

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def header_functions():
    text = open(os.path.join(ROOT, "include", "rpa.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(rpa_[a-z_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol(pkg):
    lib = pkg._lib.load()
    names = header_functions()
    assert set(names) == set(pkg._lib.EXPORTED_SYMBOLS)
    for n in names:
        assert hasattr(lib, n), n
    assert lib.rpa_version() == 100


def test_header_links_from_two_translation_units(tmp_path):
    """A consumer with several translation units (C or C++) must link: the header may define no
    object, only types and declarations."""
    import subprocess

    inc = os.path.join(ROOT, "include")
    for cc, ext in (("gcc", "c"), ("g++", "cc")):
        a, b = tmp_path / f"a.{ext}", tmp_path / f"b.{ext}"
        a.write_text('#include "rpa.h"\nint from_a(void) { RpaMaskMode m = RPA_MASK_CUSTOM; return (int)m + RPA_VERSION; }\n')
        b.write_text('#include "rpa.h"\nint from_a(void);\nint main(void) { RpaLayout l = RPA_LAYOUT_SPLIT; '
                     'return from_a() + (int)l + (int)sizeof(RpaParams) == 0; }\n')
        out = tmp_path / f"two_units_{ext}"
        r = subprocess.run([cc, "-Wall", "-Werror", "-I", inc, str(a), str(b), "-o", str(out)],
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        assert subprocess.run([str(out)]).returncode == 0


def test_library_exports_nothing_but_the_declared_entry_points(pkg):
    """The library is built with hidden visibility: its dynamic symbol table holds the functions rpa.h
    declares and nothing else (no data object, no C++ helper a host process could collide with or interpose)."""
    import subprocess

    r = subprocess.run(["nm", "-D", "--defined-only", pkg._lib.LIB_PATH], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    defined = {}
    for ln in r.stdout.splitlines():
        parts = ln.split()
        if len(parts) == 3:
            defined[parts[2]] = parts[1]
    stray = {n: k for n, k in defined.items() if n not in header_functions() and not n.startswith("__hip_")}
    assert not stray, stray
    assert all(defined[n] == "T" for n in header_functions())


def test_measurement_library_exports_its_three_kernels(pkg):
    """lib/librpa_ceilings.so (bench.py --ceilings) is a library of its own: three launchers, nothing else."""
    import subprocess

    path = os.path.join(os.path.dirname(pkg._lib.LIB_PATH), "librpa_ceilings.so")
    assert os.path.exists(path), "build it with __graft_entry__.build()"
    r = subprocess.run(["nm", "-D", "--defined-only", path], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    names = {ln.split()[2] for ln in r.stdout.splitlines() if len(ln.split()) == 3 and not ln.split()[2].startswith("__hip_")}
    assert names == {"rpa_ceiling_stream_read", "rpa_ceiling_lds_dma_read", "rpa_ceiling_mfma"}, names


def _header_struct_fields(name):
    """Field names of a struct of rpa.h, in declaration order, read from the header's text."""
    text = open(os.path.join(ROOT, "include", "rpa.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    body = re.search(r"typedef struct %s \{(.*?)\} %s;" % (name, name), text, flags=re.S).group(1)
    fields = []
    for decl in body.split(";"):
        decl = decl.strip()
        if decl:
            fields.append(re.search(r"([A-Za-z_][A-Za-z0-9_]*)$", decl).group(1))
    return fields


@pytest.mark.parametrize("struct", ["RpaParams", "RpaMlaParams"])
def test_struct_layout_matches_header(pkg, tmp_path, struct):
    """sizeof and every offsetof as the C compiler lays the header's struct out, against the ctypes mirror:
    a field reordered or retyped on one side only fails here even when the total size stays the same."""
    import subprocess

    fields = _header_struct_fields(struct)
    mirror = getattr(pkg._lib, struct)
    assert fields == [f[0] for f in mirror._fields_]
    src = tmp_path / "layout.c"
    lines = ['#include <stdio.h>', '#include <stddef.h>', '#include "rpa.h"', "int main(void) {",
             '  printf("sizeof %%zu\\n", sizeof(%s));' % struct]
    for f in fields:
        lines.append('  printf("%s %%zu %%zu\\n", offsetof(%s, %s), sizeof(((%s*)0)->%s));' % (f, struct, f, struct, f))
    lines += ["  return 0;", "}"]
    src.write_text("\n".join(lines) + "\n")
    exe = tmp_path / "layout"
    r = subprocess.run(["gcc", "-Wall", "-Werror", "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True).stdout.split("\n")
    assert int(out[0].split()[1]) == ctypes.sizeof(mirror)
    for ln in out[1:]:
        if ln:
            name, off, size = ln.split()
            assert getattr(mirror, name).offset == int(off), name
            assert getattr(mirror, name).size == int(size), name


def base_params(pkg):
    p = pkg._lib.RpaParams()
    for f in ("q", "out", "kv_cache", "kv_lens", "page_indices", "cu_q_lens", "cu_kv_lens"):
        setattr(p, f, 0x1000)  # never dereferenced by the validators
    p.num_tokens, p.num_seqs, p.num_q_heads, p.num_kv_heads = 8, 3, 8, 2
    p.head_dim, p.page_size, p.total_pages = 128, 4, 16
    p.decode_end = 1
    p.sm_scale = 1.0
    return p


def test_a_caller_of_the_earlier_struct_is_read_no_further_than_it_reaches(pkg):
    """RpaParams grew two fields behind `distribution`: they are read where the layout says that they are there, else taken as
    0 whatever lies behind the caller's struct."""
    lib, tail = pkg._lib.load(), pkg._lib.RPA_PARAMS_TAIL
    P = pkg._lib.RpaParams
    old_size = P.q_head_dim.offset
    assert old_size == P.distribution.offset + 8

    def answers(p):
        buf = ctypes.create_string_buffer(1024)
        ref = ctypes.cast(ctypes.addressof(p), ctypes.POINTER(P))
        n = lib.rpa_describe_plan(ref, buf, len(buf))
        return lib.rpa_validate(ref), lib.rpa_workspace_bytes(ref), lib.rpa_mask_needs_starts(ref), n, buf.value

    for layout in (pkg._lib.RPA_LAYOUT_FUSED, pkg._lib.RPA_LAYOUT_SPLIT):
        p = base_params(pkg)
        p.layout, p.v_pages = layout, 0x1000
        want = answers(p)
        assert want[0] == 0 and want[3] > 0
        for rest in (b"\xff" * 64, b"\x40\0\0\0\x01\0\0\0" * 8):  # -1, -1, ...; 64, 1, ...
            assert answers(ctypes.create_string_buffer(bytes(p)[:old_size] + rest)) == want
        # the same fields where the caller says that they are there
        p.layout = layout | tail
        assert answers(p) == want
        p.q_head_dim = -1
        assert status(pkg, lib.rpa_validate(ctypes.byref(p))) == "RPA_EUNSUPPORTED"
        p.q_head_dim = 64
        assert lib.rpa_validate(ctypes.byref(p)) == 0
    for layout in (2, 0x102, 0x200, -1):
        p.layout = layout
        assert status(pkg, lib.rpa_validate(ctypes.byref(p))) == "RPA_EINVAL_SHAPE"


@pytest.mark.parametrize("D,tokens", [(128, 1), (128, 64), (128, 65), (256, 4)])
def test_a_call_without_sequences_launches_nothing(pkg, D, tokens):
    """A bucket of no sequences, composition on the device: its arrays may have no element, so nothing may be launched that reads the
    first one's lengths.  (Without a GPU a launch is an error; with one the addresses below would be read.)"""
    import torch

    if torch.cuda.device_count() > 0:
        pytest.skip("a launch is seen by its failing without a GPU")
    lib = pkg._lib.load()
    for lens in (0x1000, None):
        p = base_params(pkg)
        p.num_seqs, p.num_tokens, p.decode_end, p.head_dim = 0, tokens, 0, D
        p.distribution, p.kv_lens, p.page_indices, p.max_kv_len = 0x1000, lens, lens, 100
        assert lib.rpa_workspace_bytes(ctypes.byref(p)) == 0
        for new in (None, 0x1000):
            assert lib.rpa_attention_update(ctypes.byref(p), new, new, None) == 0
        assert lib.rpa_decode(ctypes.byref(p), None) == 0
        assert lib.rpa_prefill(ctypes.byref(p), None) == 0


def status(pkg, code):
    return pkg._lib.STATUS_NAMES[code]


def test_static_validation_codes(pkg):
    lib = pkg._lib.load()
    p = base_params(pkg)
    assert lib.rpa_validate(ctypes.byref(p)) == 0
    p.num_q_heads = 7
    assert status(pkg, lib.rpa_validate(ctypes.byref(p))) == "RPA_EINVAL_HEADS"
    assert b"divisible" in lib.rpa_last_error()
    p = base_params(pkg); p.sliding_window = -1
    assert status(pkg, lib.rpa_validate(ctypes.byref(p))) == "RPA_EINVAL_WINDOW"
    p = base_params(pkg); p.kv_dtype = 5
    assert status(pkg, lib.rpa_validate(ctypes.byref(p))) == "RPA_EINVAL_DTYPE"
    p = base_params(pkg); p.decode_end = 4
    assert status(pkg, lib.rpa_validate(ctypes.byref(p))) == "RPA_EINVAL_DISTRIBUTION"
    p = base_params(pkg); p.head_dim = 64
    assert status(pkg, lib.rpa_validate(ctypes.byref(p))) == "RPA_EUNSUPPORTED"
    # 256-wide heads: accepted (q_scale too), no workspace for short rows
    p = base_params(pkg); p.head_dim = 256
    assert lib.rpa_validate(ctypes.byref(p)) == 0
    p.decode_end = p.num_seqs
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == 0
    p.q_scale = 0.5
    assert lib.rpa_validate(ctypes.byref(p)) == 0
    p = base_params(pkg); p.softmax_dtype = 7
    assert status(pkg, lib.rpa_validate(ctypes.byref(p))) == "RPA_EINVAL_DTYPE"
    p = base_params(pkg); p.q_scale = -1.0
    assert status(pkg, lib.rpa_validate(ctypes.byref(p))) == "RPA_EINVAL_SHAPE"
    p = base_params(pkg); p.q = None
    assert status(pkg, lib.rpa_validate(ctypes.byref(p))) == "RPA_EINVAL_NULL"
    p = base_params(pkg); p.layout = 1
    assert status(pkg, lib.rpa_validate(ctypes.byref(p))) == "RPA_EINVAL_NULL"  # split layout without v_pages
    assert lib.rpa_validate(None) == -12


def host_check(pkg, p, kv_lens, pages, cu_q, cu_kv, dist):
    lib = pkg._lib.load()
    arr = lambda a: None if a is None else np.ascontiguousarray(a, dtype=np.int32)
    a = [arr(x) for x in (kv_lens, pages, cu_q, cu_kv, dist)]
    ptr = lambda x: None if x is None else x.ctypes.data_as(ctypes.POINTER(ctypes.c_int32))
    rc = lib.rpa_validate_host(ctypes.byref(p), ptr(a[0]), ptr(a[1]), len(a[1]), ptr(a[2]), ptr(a[3]), ptr(a[4]))
    return pkg._lib.STATUS_NAMES[rc], lib.rpa_last_error().decode()


def test_dynamic_validation_codes(pkg):
    p = base_params(pkg)
    kv, cu_q, cu_kv = [5, 8, 6], [0, 1, 4, 8], [0, 8, 16, 24]
    pages = [1, 2, 3, 4, 5, 6]
    ok = host_check(pkg, p, kv, pages, cu_q, cu_kv, [1, 1, 3])
    assert ok[0] == "RPA_OK", ok
    assert host_check(pkg, p, kv, pages, cu_q, cu_kv, [2, 1, 3])[0] == "RPA_EINVAL_DISTRIBUTION"
    # q_len > kv_len (message of ragged_paged_attention_v3.py:1475-1476)
    st, msg = host_check(pkg, p, [5, 2, 6], pages, cu_q, cu_kv, [1, 1, 3])
    assert st == "RPA_EINVAL_QLEN_GT_KVLEN" and "q_len=3 > kv_len=2" in msg
    # q_len == 0
    assert host_check(pkg, p, kv, pages, [0, 1, 1, 8], cu_kv, [1, 1, 3])[0] == "RPA_EINVAL_QLEN_GT_KVLEN"
    # page index out of range
    st, msg = host_check(pkg, p, kv, [1, 2, 3, 16, 5, 6], cu_q, cu_kv, [1, 1, 3])
    assert st == "RPA_EINVAL_PAGE_RANGE" and "out of [0, 16)" in msg
    assert host_check(pkg, p, kv, [1, 2, -1, 4, 5, 6], cu_q, cu_kv, [1, 1, 3])[0] == "RPA_EINVAL_PAGE_RANGE"
    # page list runs off the end of page_indices
    assert host_check(pkg, p, kv, pages[:5], cu_q, cu_kv, [1, 1, 3])[0] == "RPA_EINVAL_PAGE_RANGE"
    # tokens exceed T
    assert host_check(pkg, p, [5, 8, 9], pages + [7], [0, 1, 4, 9], [0, 8, 16, 28], [1, 1, 3])[0] == "RPA_EINVAL_SHAPE"
    # decode row with q_len 2
    assert host_check(pkg, p, kv, pages, [0, 2, 4, 8], cu_kv, [1, 1, 3])[0] == "RPA_EINVAL_DISTRIBUTION"
    # padded 2-D table: page_cnt > pages_per_seq
    p2 = base_params(pkg); p2.cu_kv_lens = None; p2.pages_per_seq = 1
    st, msg = host_check(pkg, p2, kv, [1, 2, 3], cu_q, None, [1, 1, 3])
    assert st == "RPA_EINVAL_PAGE_RANGE" and "pages_per_seq=1" in msg


def test_workspace_size_is_deterministic(pkg):
    lib = pkg._lib.load()
    p = base_params(pkg)
    p.num_seqs = p.decode_end = 16
    p.num_tokens = 16
    p.num_q_heads, p.num_kv_heads, p.page_size, p.total_pages = 32, 8, 64, 8192
    p.max_kv_len = 32768
    # lengths unknown to the host: the balanced plan, two groups of 16 partial rows per wave slot
    # plus the prefix sum of blocks (17 words, padded to 8 bytes) and one 8-byte arrival word per
    # (row, unit, wave): 16 rows x 2 units x 4 waves; its size does not depend on the batch
    a = lib.rpa_workspace_bytes(ctypes.byref(p))
    assert a > 0 and a == lib.rpa_workspace_bytes(ctypes.byref(p))
    assert (a - 18 * 4 - 16 * 2 * 4 * 8) % (2 * 16 * 130 * 4) == 0
    p.max_kv_len = 8192
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == a
    # all rows of one known length: the fixed plan, one partial row per (row, split, head)
    p.max_kv_len = 32768
    p.sum_decode_kv_len = 16 * 32768
    f = lib.rpa_workspace_bytes(ctypes.byref(p))
    assert f > 0 and f % (16 * 32 * 130 * 4) == 0
    p.num_splits = 1
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == 0


def test_workspace_for_prefill_launches_that_leave_the_gpu_idle(pkg, monkeypatch):
    """rpa_workspace_bytes also reports the room that lets an under-filled prefill launch cut its K/V
    ranges into pieces: (tokens x heads x pieces) partial rows of 128 + 2 floats.  Nothing for launches
    that fill the GPU, for calls whose composition is on the device, without a bound on the lengths,
    or with RPA_PREFILL_SPLITS=0; the forced count is honoured."""
    lib = pkg._lib.load()
    monkeypatch.delenv("RPA_PREFILL_SPLITS", raising=False)

    def params(tokens, hq, hkv, max_kv):
        p = base_params(pkg)
        p.num_seqs, p.decode_end, p.num_tokens = 1, 0, tokens
        p.num_q_heads, p.num_kv_heads, p.page_size, p.total_pages = hq, hkv, 64, 8192
        p.max_q_len, p.max_kv_len = tokens, max_kv
        return p

    row = (128 + 2) * 4
    p = params(512, 8, 2, 16384)  # one 512-token chunk on a long prefix, 32 workgroups
    need = lib.rpa_workspace_bytes(ctypes.byref(p))
    assert need > 0 and need % (512 * 8 * row) == 0
    pieces = need // (512 * 8 * row)
    assert 2 <= pieces <= 64
    p.max_kv_len = 0  # no bound on the lengths: no cut
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == 0
    p = params(512, 8, 2, 16384)
    p.distribution = 0x1000  # composition on the device: the same rule on the bounds (every workgroup fits the count to its range)
    monkeypatch.setenv("RPA_PREFILL_SPLITS", "0")
    dyn = lib.rpa_workspace_bytes(ctypes.byref(p))  # what the decode plan of such a call asks for
    monkeypatch.setenv("RPA_PREFILL_SPLITS", "7")
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == max(dyn, 512 * 8 * 7 * row)
    monkeypatch.delenv("RPA_PREFILL_SPLITS")
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == max(dyn, need)
    p = params(2048, 32, 8, 8192)  # 512 workgroups: the GPU is full
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == 0
    p = params(1000, 8, 4, 1000)  # a short range: the merge would cost what the cut saves
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == 0
    p = params(16, 8, 2, 32768)  # a verify step on a long context: the short-chunk tile, many pieces
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) // (16 * 8 * row) >= 16
    p.kv_dtype = 1  # e4m3 caches take the compiled kernels (128 positions per workgroup), which cut too
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) // (16 * 8 * row) >= 16
    p = params(200, 4, 1, 3000)  # 256-wide heads: rows of 256 + 2 floats
    p.head_dim = 256
    need = lib.rpa_workspace_bytes(ctypes.byref(p))
    assert need > 0 and need % (200 * 4 * (256 + 2) * 4) == 0
    p = params(512, 8, 2, 16384)
    monkeypatch.setenv("RPA_PREFILL_SPLITS", "0")
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == 0
    monkeypatch.setenv("RPA_PREFILL_SPLITS", "5")
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == 512 * 8 * 5 * row


def test_workspace_for_a_custom_mask_as_bits(pkg, monkeypatch):
    """Custom masks: rpa_workspace_bytes adds one bit per (query token, kv token up to the bound on the lengths),
    rows of whole 64-bit words, behind the partial rows of a cut launch (256-byte aligned).  Not without a bound on
    the lengths, not for 256-wide heads, not with RPA_MASK_BITS=0."""
    lib = pkg._lib.load()
    monkeypatch.delenv("RPA_PREFILL_SPLITS", raising=False)
    monkeypatch.delenv("RPA_MASK_BITS", raising=False)
    p = base_params(pkg)
    p.num_seqs, p.decode_end, p.num_tokens = 64, 0, 1024
    p.num_q_heads, p.num_kv_heads, p.page_size, p.total_pages = 32, 8, 64, 8192
    p.max_q_len, p.max_kv_len = 16, 4112
    p.mask_mode = 1
    p.custom_mask = 0x1000
    p.cu_mask_lens = 0x1000
    bits = 1024 * ((4112 + 63) // 64) * 8
    monkeypatch.setenv("RPA_PREFILL_SPLITS", "0")
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == bits
    monkeypatch.setenv("RPA_PREFILL_SPLITS", "3")
    partial = 1024 * 32 * 3 * (128 + 2) * 4
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == ((partial + 255) // 256) * 256 + bits
    monkeypatch.setenv("RPA_MASK_BITS", "0")
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == partial
    monkeypatch.delenv("RPA_MASK_BITS")
    monkeypatch.setenv("RPA_PREFILL_SPLITS", "0")
    p.max_kv_len = 0
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == 0
    p.max_kv_len = 4112
    p.head_dim = 256
    assert lib.rpa_workspace_bytes(ctypes.byref(p)) == 0


def test_python_wrapper_raises_like_the_reference(pkg):
    import torch

    q = torch.zeros(4, 8, 128, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no CPU path"):
        pkg.ragged_paged_attention(q, None, None, torch.zeros(2, 4, 4, 128, dtype=torch.bfloat16),
                                   torch.zeros(2, dtype=torch.int32), torch.zeros(2, dtype=torch.int32),
                                   torch.zeros(3, dtype=torch.int32), torch.zeros(3, dtype=torch.int32), [0, 0, 2], None)
    m = __import__("sglang_jax_amd.ragged_paged_attention", fromlist=["x"])
    i32 = lambda *s: torch.zeros(*s, dtype=torch.int32)
    cache = torch.zeros(2, 4, 4, 128, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="must be positive"):
        m.static_validate_inputs(q, None, None, cache, i32(2), i32(2), i32(3), i32(3), i32(3), sliding_window=0)
    with pytest.raises(ValueError, match="must not be 0.0"):
        m.static_validate_inputs(q, None, None, cache, i32(2), i32(2), i32(3), i32(3), i32(3), soft_cap=0.0)
    with pytest.raises(ValueError, match="divisible"):
        m.static_validate_inputs(q, None, None, torch.zeros(2, 4, 6, 128, dtype=torch.bfloat16), i32(2), i32(2), i32(3),
                                 i32(3), i32(3))
    with pytest.raises(ValueError, match=r"cu_q_lens.shape"):
        m.static_validate_inputs(q, None, None, cache, i32(2), i32(2), i32(4), i32(3), i32(3))
    with pytest.raises(ValueError, match="int32"):
        m.static_validate_inputs(q, None, None, cache, torch.zeros(2, dtype=torch.int64), i32(2), i32(3), i32(3), i32(3))
    with pytest.raises(ValueError, match="Expected 3D"):
        m.static_validate_inputs(q, torch.zeros(4, 2), torch.zeros(4, 2), cache, i32(2), i32(2), i32(3), i32(3), i32(3))


def test_generated_assembly_is_up_to_date(tmp_path):
    """The generated include files (the assembly loops of the prefill and MLA kernels) are what
    their generators write today, with no experiment switch set."""
    import shutil
    import subprocess

    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sglang-jax_amd", "csrc")
    work = tmp_path / "csrc"
    work.mkdir()
    for name in ("gen_prefill_pipe_loop.py", "gen_mla_pipe_loop.py", "gen_mla_wide_loop.py", "gen_mla_wide32_loop.py"):
        shutil.copy(os.path.join(csrc, name), work / name)
    env = {k: v for k, v in os.environ.items() if not k.startswith(("RPA_PIPE_", "RPA_MLA_PIPE_", "RPA_MLA_WIDE_"))}
    env["PYTHONDONTWRITEBYTECODE"] = "1"
    for gen, inc in (("gen_prefill_pipe_loop.py", "rpa_prefill_pipe_loop.inc"), ("gen_mla_pipe_loop.py", "rpa_mla_pipe_loop.inc"),
                     ("gen_mla_wide_loop.py", "rpa_mla_wide_loop.inc"), ("gen_mla_wide32_loop.py", "rpa_mla_wide32_loop.inc")):
        subprocess.run([sys.executable, str(work / gen)], check=True, env=env, stdout=subprocess.DEVNULL)
        with open(work / inc) as f, open(os.path.join(csrc, inc)) as g:
            assert f.read() == g.read(), f"{inc} is stale: run {gen}"


def _device_code():
    """The device code objects of the built library, as files."""
    import struct
    import tempfile

    with open(os.path.join(ROOT, "sglang-jax_amd", "lib", "librpa_mi355.so"), "rb") as f:
        blob = f.read()
    at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        (n,), pos = struct.unpack_from("<Q", blob, at + 24), at + 32
        for _ in range(n):
            offset, size, name_len = struct.unpack_from("<QQQ", blob, pos)
            target = blob[pos + 24 : pos + 24 + name_len]
            pos += 24 + name_len
            if not size or b"gfx950" not in target:
                continue
            with tempfile.NamedTemporaryFile(suffix=".co") as co:
                co.write(blob[at + offset : at + offset + size])
                co.flush()
                yield co.name
        at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 1)


def _llvm(tool, *args):
    import subprocess

    path = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", tool)
    return subprocess.run([path, *args], check=True, capture_output=True, text=True).stdout


def _device_kernels():
    """{demangled kernel name: (spilled vector registers, scratch bytes per lane)} of the built library, from the metadata
    notes of its device code."""
    import subprocess

    found = {}
    for co in _device_code():
        for entry in _llvm("llvm-readelf", "--notes", co).split(".agpr_count")[1:]:
            value = {k: re.search(rf"\.{k}:\s+(\S+)", entry).group(1) for k in ("symbol", "vgpr_spill_count", "private_segment_fixed_size")}
            found[value["symbol"]] = (int(value["vgpr_spill_count"]), int(value["private_segment_fixed_size"]))
    names = subprocess.run(["c++filt"], input="\n".join(n.removesuffix(".kd") for n in found), capture_output=True, text=True, check=True).stdout.split("\n")
    return dict(zip(names, found.values()))


def test_decode_kernels_keep_their_block_loops_in_registers(pkg):
    """A spilled register in a decode kernel's block loop is a reload that waits for the K/V loads in flight.  The kernels of
    whole rows and of fixed pieces have none, with and without the general score path (soft cap, rounded logits), on either
    kind of pages; the balanced kernels as many as are listed (in-kernel merge; soft cap on whole pages)."""
    kernels = {k: v for k, v in _device_kernels().items() if "rpa_decode_" in k or "rpa_rows256_kernel" in k}
    assert len(kernels) >= 40
    spilled = {re.search(r"rpa_\w+(<.*?>)?", k).group(0): v[0] for k, v in kernels.items() if v[0]}
    # <MT, FP8, UNIFORM_PAGE, CAP, in-kernel merge, HALF>
    allowed = {"rpa_decode_balanced_kernel<1, false, false, false, true, false>": 4,
               "rpa_decode_balanced_kernel<1, false, false, true, true, false>": 4,
               "rpa_decode_balanced_kernel<1, false, true, false, true, false>": 4,
               "rpa_decode_balanced_kernel<1, false, true, true, true, false>": 9,
               "rpa_decode_balanced_kernel<1, false, true, true, false, false>": 4}
    assert all(n <= allowed.get(k, 0) for k, n in spilled.items()), spilled


def _instructions():
    """(kernel, [(operation, operands), ...]) of the built library's device code, in program order."""
    for co in _device_code():
        kernel, ins = None, []
        for line in _llvm("llvm-objdump", "-d", "--no-show-raw-insn", "--no-leading-addr", co).split("\n"):
            if line.startswith("<") and line.endswith(">:"):
                if ins:
                    yield kernel, ins
                kernel, ins = line[1:-2], []
            elif line.startswith("\t"):
                operation, _, operands = line.split("//")[0].strip().partition(" ")
                ins.append((operation, operands))
        if ins:
            yield kernel, ins


def _vector_registers(operand):
    m = re.match(r"v\[(\d+):(\d+)\]|v(\d+)", operand.strip())
    return set() if not m else {int(m.group(3))} if m.group(3) else set(range(int(m.group(1)), int(m.group(2)) + 1))


def test_a_wide_store_keeps_its_data(pkg):
    """A store of more than 8 bytes reads its registers after it has issued: one wait state before a vector instruction writes them.
    The compiler keeps it behind its own stores; those of inline assembly (written through, sc1) bring it along."""
    written_through, overwritten, bare = 0, [], []
    for kernel, ins in _instructions():
        for (op, operands), (then, target) in zip(ins, ins[1:]):
            if not re.match(r"(global|flat|scratch|buffer)_store_dwordx[34]$", op):
                continue
            fields = re.split(r",\s*(?![^\[]*\])", operands)
            data = _vector_registers(fields[0 if op.startswith("buffer") else 1])
            by_scalar = op.startswith("buffer") and re.match(r"s\d", fields[3])  # a scalar offset is that wait state
            if then.startswith("v_") and not by_scalar and data & _vector_registers(target):
                overwritten.append((kernel, operands, then, target))
            if op.startswith("global") and "sc1" in operands:
                written_through += 1
                if then != "s_nop":
                    bare.append((kernel, operands, then))
    assert written_through > 0
    assert not overwritten and not bare, (overwritten[:3], bare[:3])


def test_a_copy_into_lds_finds_its_address(pkg):
    """A copy into LDS takes its address from m0, which a scalar instruction has to have written one wait state before: another
    instruction, or s_nop, stands in between.  (All of these copies are inline assembly, which the compiler does not look into.)"""
    copies, short = 0, []
    for kernel, ins in _instructions():
        for (op, operands), (then, target) in zip(ins, ins[1:]):
            if "_load_lds_" in then:
                copies += 1
                if op.startswith("s_") and operands.split(",")[0] == "m0":
                    short.append((kernel, op, operands, then, target))
    assert copies > 1000
    assert not short, (len(short), short[:3])


def _scalar_registers(operands):
    found = set()
    for lo, hi, one in re.findall(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b", operands):
        found |= {int(one)} if one else set(range(int(lo), int(hi) + 1))
    return found | ({"vcc"} if "vcc" in operands else set())


def test_a_memory_instruction_finds_its_scalars(pkg):
    """A scalar register that a vector instruction wrote (v_readfirstlane) is read by a memory instruction no sooner than five wait states
    later: what stands between counts one each, s_nop n counts n + 1.  The compiler keeps that for its own instructions, inline assembly
    has to keep it by itself, whatever the compiler puts in front."""
    readers, short = 0, []
    for kernel, ins in _instructions():
        written = {}  # scalar register -> wait states since a vector instruction wrote it
        for op, operands in ins:
            if re.match(r"(global|buffer|flat|scratch)_", op):
                read = _scalar_registers(operands)
                readers += bool(read)
                if any(written.get(r, 5) < 5 for r in read):
                    short.append((kernel, op, operands))
            states = int(operands.split()[0], 0) + 1 if op == "s_nop" else 1
            written = {r: n + states for r, n in written.items() if n + states < 5}
            fields = re.split(r",\s*(?![^\[]*\])", operands)
            if op.startswith("v_"):  # (carries and comparisons: the second operand, or the first)
                wrote = _scalar_registers(fields[0])
                if re.match(r"v_(add|sub|subrev|addc|subb|subbrev)_co|v_div_scale|v_mad_[iu]64", op) and len(fields) > 1:
                    wrote |= _scalar_registers(fields[1])
                written.update({r: 0 for r in wrote})
            elif op.startswith("s_") and not re.match(r"s_(cmp|bitcmp|set|nop|wait)", op):
                for r in _scalar_registers(fields[0]):  # (written anew by a scalar instruction)
                    written.pop(r, None)
    assert readers > 1000
    assert not short, (len(short), short[:3])


def test_bases_of_latent_tiles_are_worked_out_by_scalar_instructions(pkg):
    """Where a tile begins is the same for all lanes, and the MLA kernels keep it known to the compiler: no copy's scalar base comes back
    from vector registers (a row length read from LDS made every address of the sparse kernels the lane's own)."""
    copies, returned = 0, []
    for kernel, ins in _instructions():
        from_lanes = set()
        for op, operands in ins if "mla" in kernel else ():
            if "_load_lds_" in op and (base := _scalar_registers(operands)):
                copies += 1
                if base & from_lanes:
                    returned.append((kernel, operands))
            first = _scalar_registers(operands.split(",")[0])
            if op.startswith(("v_readfirstlane", "v_readlane")):
                from_lanes |= first
            elif op.startswith("s_") and not re.match(r"s_(cmp|bitcmp|set|nop|wait)", op):
                from_lanes -= first
    assert copies > 1000
    assert not returned, (len(returned), returned[:3])


# ------------------------------------------------------------------ the shape table (csrc/rpa_shapes.h)
def _shape_params(pkg, *, S, decode_end, T, Hq, Hkv, D=128, P=64, fp8=False, max_q=0, max_kv=0, sum_dec=0, **opts):
    p = base_params(pkg)
    p.num_tokens, p.num_seqs, p.num_q_heads, p.num_kv_heads = T, S, Hq, Hkv
    p.head_dim, p.page_size, p.total_pages = D, P, 1 << 20
    p.decode_end, p.max_q_len, p.max_kv_len, p.sum_decode_kv_len = decode_end, max_q, max_kv, sum_dec
    p.kv_dtype = pkg._lib.RPA_KV_FP8_E4M3 if fp8 else pkg._lib.RPA_KV_BF16
    for k, v in opts.items():
        setattr(p, k, v)
    return p


def test_shape_table_rows_of_the_benchmark_configurations(pkg):
    """rpa_describe_plan: which row of the shape table, which kernel and which split plan a call takes (the
    reference answers the same question with get_tuned_block_sizes, tuned_block_sizes_v3.py:2163-2229).
    The five benchmark shapes and the option / head-width / chunk-length branches of the table."""
    d = pkg._lib.describe_plan
    c1 = d(_shape_params(pkg, S=8, decode_end=8, T=8, Hq=16, Hkv=8, P=16, max_kv=512, sum_dec=2300))
    assert "shape=decode_bf16_small" in c1 and "rpa_decode_splitkv_kernel" in c1 and "waves_per_wg=2" in c1
    assert "prefill" not in c1
    c2 = d(_shape_params(pkg, S=64, decode_end=56, T=8760, Hq=32, Hkv=8, max_q=2048, max_kv=4096, sum_dec=130000))
    assert "shape=decode_bf16_stream kernel=rpa_decode_balanced_kernel rows=56 waves_per_wg=4 resident_waves=1024" in c2
    assert "shape=prefill_pipe kernel=rpa_prefill_pipe_kernel tile=128x1x64 kv_pieces_with_workspace=1" in c2
    c3 = d(_shape_params(pkg, S=16, decode_end=16, T=16, Hq=32, Hkv=8, max_kv=32768, sum_dec=16 * 32768))
    assert "shape=decode_bf16_stream kernel=rpa_decode_splitkv_kernel" in c3 and "merge=rpa_combine_kernel" in c3
    c4 = d(_shape_params(pkg, S=128, decode_end=128, T=128, Hq=64, Hkv=8, fp8=True, max_kv=8192, sum_dec=590000))
    assert "shape=decode_fp8_stream kernel=rpa_decode_balanced_kernel" in c4 and "resident_waves=1024" in c4
    # chunks of at most 64 tokens with heads in fours: the short-chunk tile; a long prompt on few heads is cut
    short = d(_shape_params(pkg, S=64, decode_end=0, T=1024, Hq=32, Hkv=8, max_q=16, max_kv=4096))
    assert "shape=prefill_pipe_short" in short and "tile=32x4x64" in short
    one = d(_shape_params(pkg, S=1, decode_end=0, T=16, Hq=8, Hkv=2, max_q=16, max_kv=32768))
    assert "kv_pieces_with_workspace=1 " not in one  # an under-filled launch cuts its K/V range
    # options and cache types leave the assembly kernel
    assert "shape=prefill_options kernel=rpa_prefill_async_kernel" in d(_shape_params(
        pkg, S=2, decode_end=0, T=600, Hq=32, Hkv=8, max_q=300, max_kv=600, soft_cap=30.0))
    assert "shape=prefill_fp8 kernel=rpa_prefill_staged_kernel" in d(_shape_params(
        pkg, S=2, decode_end=0, T=600, Hq=32, Hkv=8, max_q=300, max_kv=600, fp8=True))
    assert "shape=prefill_pipe " not in d(_shape_params(pkg, S=2, decode_end=0, T=600, Hq=32, Hkv=8, P=48, max_q=300, max_kv=600))
    wide = d(_shape_params(pkg, S=6, decode_end=4, T=304, Hq=16, Hkv=4, D=256, max_q=200, max_kv=900, sum_dec=3000))
    assert "shape=decode_256 kernel=rpa_rows256_kernel" in wide and "shape=prefill_256 kernel=rpa_prefill_async_kernel" in wide


def test_described_plan_names_what_runs(pkg):
    """The kernels of a whole call beside those of its partitions, the 256-wide prefill kernel by its name, and who leaves
    the new tokens in the cache."""
    d, tail = pkg._lib.describe_plan, pkg._lib.RPA_PARAMS_TAIL
    wide = d(_shape_params(pkg, S=6, decode_end=4, T=304, Hq=16, Hkv=4, D=256, max_q=200, max_kv=900, sum_dec=3000))
    assert "kernel=rpa_prefill_async_kernel_wide " in wide and "whole call" not in wide
    # decode rows only: their kernels write the tokens; with chunks behind them, or 256-wide heads and more than 768 MB, a launch in front does
    rows = dict(S=64, decode_end=64, T=64, Hq=32, Hkv=8, max_kv=4000, sum_dec=130000)
    assert d(_shape_params(pkg, **rows)).endswith("new tokens: written by the decode kernels\n")
    assert "written by rpa_kv_write_kernel, in front" in d(_shape_params(pkg, D=256, **rows))
    assert d(_shape_params(pkg, D=256, **{**rows, "sum_dec": 90000})).endswith("new tokens: written by the decode kernels\n")
    assert d(_shape_params(pkg, D=256, sliding_window=1024, **rows)).endswith("new tokens: written by the decode kernels\n")
    mixed = dict(S=64, decode_end=56, T=8760, Hq=32, Hkv=8, max_q=2048, max_kv=4096, sum_dec=130000)
    assert "written by rpa_kv_write_kernel, in front" in d(_shape_params(pkg, **mixed))
    bucket = d(_shape_params(pkg, distribution=0x1000, **mixed))
    assert "the decode kernels, those of chunks by rpa_kv_write_kernel" in bucket and "whole call" not in bucket
    # a few query tokens on short contexts: rows of the decode kernels, chunk or not
    few = d(_shape_params(pkg, S=3, decode_end=1, T=20, Hq=16, Hkv=8, P=16, max_q=12, max_kv=500, sum_dec=300))
    assert few.startswith("whole call: shape=decode_bf16_stream kernel=rpa_decode_splitkv_kernel rows=20 ")
    assert "\nprefill: shape=prefill_options" in few and few.endswith("written by the decode kernels\n")
    # prompts without a prefix read the caller's rows; the kernel is that of the cache's pages all the same
    prompt = dict(S=1, decode_end=0, T=1003, Hq=8, Hkv=2, max_q=1003, max_kv=1003, prompts_only=1)
    for P, kernel in ((64, "shape=prefill_pipe kernel=rpa_prefill_pipe_kernel"), (16, "shape=prefill_options kernel=rpa_prefill_async_kernel "),
                      (96, "shape=prefill_options kernel=rpa_prefill_async_kernel ")):
        text = d(_shape_params(pkg, P=P, layout=tail, **prompt))
        assert kernel in text and "written by workgroups of the prefill launch, which reads the caller's rows" in text
        text = d(_shape_params(pkg, P=P, **prompt))  # (the promise is not read without the flag)
        assert kernel in text and "written by rpa_kv_write_kernel, in front" in text


@pytest.mark.parametrize("chunks,longest,Hq,Hkv,opts,streams", [
    ([1900, 1980, 2020, 2048], 18432, 32, 8, {}, True), ([1024, 1000, 1020, 1010], 13000, 32, 8, dict(fp8=True), True),
    # a round and a bit of the compiled kernels: the last sequence's workgroups would be waited for
    ([1905, 321], 7716, 32, 8, dict(fp8=True), False), ([1905, 700], 7716, 32, 8, dict(fp8=True), False), ([1905, 321], 7716, 32, 8, dict(soft_cap=30.0), False),
    ([1905, 321], 7716, 32, 8, {}, True),  # the assembly kernel
    ([1905, 60], 7716, 32, 8, dict(fp8=True), True),  # all at once
    ([1905, 1200], 7716, 32, 8, dict(fp8=True), False), ([1905, 1600], 7716, 32, 8, dict(fp8=True), True),  # 1.56 and 1.75 rounds
    # fewer heads per kv head
    ([2000] * 3, 7000, 16, 8, {}, False), ([2400, 2300], 16100, 24, 8, {}, True), ([1500] * 6, 7500, 16, 8, {}, True),
    # 4608 tokens, behind a window too; one sequence; kv heads that are not in eights; 256-wide heads
    ([2000] * 4, 4607, 32, 8, {}, False), ([2000] * 4, 4608, 32, 8, {}, True), ([2000] * 4, 9000, 32, 8, dict(sliding_window=4479), False),
    ([2000] * 4, 9000, 32, 8, dict(sliding_window=4480), True), ([4000], 9000, 32, 8, {}, False), ([2000] * 4, 9000, 16, 4, {}, False),
    ([2000] * 4, 9000, 32, 8, dict(D=256), False),
])
def test_sequences_one_after_the_other_by_their_work(pkg, chunks, longest, Hq, Hkv, opts, streams):
    """The order by streams: as many workgroups as fit at once, or 5/3 of them and more; on the assembly kernel with four heads or
    more per kv head in between too."""
    text = pkg._lib.describe_plan(_shape_params(pkg, S=len(chunks), decode_end=0, T=sum(chunks), Hq=Hq, Hkv=Hkv, max_q=max(chunks),
                                                max_kv=longest, **opts))
    assert ("\nprefill, long sequences: one after the other\n" in text) == streams, text


def test_sequences_one_after_the_other_on_workgroups_of_256_rows(pkg, monkeypatch):
    """A kernel with one workgroup per CU has half the places: 384 workgroups of 256 rows are more than fit."""
    p = _shape_params(pkg, S=3, decode_end=0, T=3072, Hq=32, Hkv=8, max_q=1024, max_kv=6024)
    for rows_in_128s in ("1", "2"):
        monkeypatch.setenv("RPA_PREFILL_PIPE_NQ", rows_in_128s)
        assert "one after the other" in pkg._lib.describe_plan(p)


def test_plans_on_both_sides_of_their_rules(pkg, monkeypatch):
    """Prefill launches that the tiles of 128 positions leave idle, rows of one length in a mostly empty last round, and the
    pieces of 256-wide rows with what they need of a workspace."""
    d = pkg._lib.describe_plan

    def packed(q, Hq, Hkv, S=1, **kw):
        return "rpa_prefill_packed_kernel" in d(_shape_params(pkg, S=S, decode_end=0, T=S * q, Hq=Hq, Hkv=Hkv, max_q=q, **{"max_kv": q, **kw}))

    assert packed(1003, 8, 2) and packed(2048, 8, 2) and packed(128, 8, 2, max_kv=4000) and packed(8, 8, 4, S=16, max_kv=1000)
    assert packed(8, 64, 8, S=8, max_kv=4000) and packed(1003, 8, 2, P=16, fp8=True) and packed(1003, 8, 2, P=24)
    # the chip is full, the tile of four heads is the better, wide heads, a pinned partition, lengths on the device or unknown
    assert not packed(1003, 32, 8) and not packed(4096, 8, 2) and not packed(500, 32, 8) and not packed(1003, 8, 2, D=256)
    assert not packed(1003, 8, 2, num_splits=1) and not packed(1003, 8, 2, distribution=0x1000) and not packed(1003, 8, 2, max_kv=0)
    monkeypatch.setenv("RPA_PREFILL_PACKED", "1")
    for Hq, Hkv, P, fp8 in ((8, 2, 64, False), (2, 2, 64, False), (10, 2, 16, False), (40, 2, 24, False), (32, 1, 1, False), (6, 2, 8, True)):
        assert packed(64, Hq, Hkv, S=6, P=P, fp8=fp8, max_kv=1500), (Hq, Hkv, P, fp8)
    assert not packed(64, 33, 1, S=6, max_kv=1500)  # more heads than columns
    monkeypatch.delenv("RPA_PREFILL_PACKED")

    def rows(S, kv, **kw):
        return d(_shape_params(pkg, S=S, decode_end=S, T=S, Hq=16, Hkv=8, max_kv=kv, **{"sum_dec": S * kv, **kw})).split("\n")[0]

    # 8 waves a row on 1024 slots; from 256 MB on rows of one length leave the fixed plan below 0.7 of the rounds
    for S, balanced in ((70, True), (89, True), (90, False), (128, False), (129, True), (179, True), (180, False), (256, False)):
        assert ("rpa_decode_balanced_kernel" in rows(S, 1024)) == balanced, S
    assert "rpa_decode_splitkv_kernel" in rows(150, 400) and "pieces_per_row=1" in rows(150, 400)  # under 256 MB: whole rows
    for S, kv, pieces in ((1, 200, 4), (1, 700, 11), (8, 300, 5), (1, 30000, 118), (180, 3000, 1)):
        need = 0 if pieces == 1 else S * pieces * 16 * (256 + 2) * 4
        assert rows(S, kv, D=256).endswith(f"kernel=rpa_rows256_kernel rows={S} pieces_per_row={pieces} workspace={need}"), (S, kv)
    assert "pieces_per_row=4 " in rows(180, 3000, D=256, sum_dec=270000)  # rows that differ: twice the slots


def test_small_chunks_bring_their_tokens_where_that_is_less_work(pkg):
    """The launch of small chunks reads the new tokens from the caller's rows up to 12 M of tokens x query heads x longest chunk x bytes, on pages that are no
    multiple of a tile whatever they are; the launch in front is not counted as spared there."""
    def plan(T, q, Hq, Hkv, kv, P=64, S=2, **kw):
        d = pkg._lib.describe_plan(_shape_params(pkg, S=S, decode_end=0, T=T, Hq=Hq, Hkv=Hkv, P=P, max_q=q, max_kv=kv, **kw))
        return "rpa_prefill_packed_kernel" in d, "workgroups of the prefill launch, which reads the caller's rows" in d

    assert plan(1056, 603, 8, 2, 684) == (True, True) and plan(1170, 843, 8, 4, 881, fp8=True, P=16) == (True, True)
    assert plan(1951, 1175, 8, 1, 1512, P=128) == (True, False) and plan(1628, 1383, 8, 2, 1618, P=16) == (True, False)
    assert plan(2354, 1478, 8, 1, 1640, P=128, fp8=True) == (True, False)
    for P, beside in ((64, False), (32, False), (16, False), (48, True), (24, True)):
        assert plan(1951, 1175, 8, 1, 1512, P=P) == (True, beside), P
    for T, beside in ((1000, True), (1001, False)):
        assert plan(T, 750, 8, 1, 1512, S=2) == (True, beside), T
    assert plan(136, 74, 16, 8, 3174, P=16)[0] and not plan(136, 74, 16, 8, 3174, P=48)[0] and not plan(510, 182, 8, 4, 2894, P=48, S=3)[0]


def test_shape_table_environment_overrides(pkg, monkeypatch):
    d = pkg._lib.describe_plan
    p = _shape_params(pkg, S=64, decode_end=56, T=8760, Hq=32, Hkv=8, max_q=2048, max_kv=4096, sum_dec=130000)
    assert "rpa_prefill_pipe_kernel" in d(p)
    monkeypatch.setenv("RPA_PREFILL_PIPE", "0")  # the switches are read again whenever the environment changes
    assert "shape=prefill_options kernel=rpa_prefill_async_kernel" in d(p)
    monkeypatch.delenv("RPA_PREFILL_PIPE")
    monkeypatch.setenv("RPA_DECODE_BALANCED", "0")
    monkeypatch.setenv("RPA_DECODE_WAVES_PER_WG", "2")
    text = d(p)
    assert "rpa_decode_splitkv_kernel" in text and "waves_per_wg=2" in text and "rpa_prefill_pipe_kernel" in text
    monkeypatch.delenv("RPA_DECODE_BALANCED")
    monkeypatch.delenv("RPA_DECODE_WAVES_PER_WG")
    assert "rpa_decode_balanced_kernel" in d(p)


def _mla_params(pkg, Hq, P=64, fp8=False, S=64, T=64, max_kv=16384, sum_kv=590000, soft_cap=0.0, window=0):
    p = pkg._lib.RpaMlaParams()
    for f in ("ql_nope", "q_pe", "out", "cache_kv", "kv_lens", "page_indices", "cu_q_lens", "cu_kv_lens"):
        setattr(p, f, 0x1000)
    p.num_tokens, p.num_seqs, p.num_q_heads = T, S, Hq
    p.lkv_dim, p.rope_dim, p.page_size, p.total_pages = 512, 64, P, 1 << 16
    p.row_stride, p.rope_offset = 576, 512
    p.max_kv_len, p.sum_kv_len, p.sm_scale, p.soft_cap, p.sliding_window = max_kv, sum_kv, 0.07, soft_cap, window
    p.cache_dtype = pkg._lib.RPA_KV_FP8_E4M3 if fp8 else pkg._lib.RPA_KV_BF16
    return p


@pytest.mark.parametrize("S", [1, 4, 37, 64, 200, 256])
@pytest.mark.parametrize("Hq,fp8", [(16, False), (64, False), (128, False), (128, True)])
def test_mla_rows_of_up_to_256_tokens_are_left_whole(pkg, S, Hq, fp8):
    """Partial rows are bf16: a row that fits one piece of 256 tokens is not cut, whatever idles (nor are a few rows that a
    window clips to that); a longer one is."""
    for longest, window, most, cut in ((64, 0, 256, False), (65, 0, 256, False), (256, 0, 256, False), (4000, 225, 4, False),
                                       (2000, 0, 64, True)):
        if S > most:
            continue
        seen = min(longest, window or longest)
        for total in (S * seen, S * seen - S // 2, 0):
            d = pkg._lib.describe_mla_plan(_mla_params(pkg, Hq, fp8=fp8, S=S, T=S, max_kv=longest, sum_kv=total, window=window), False)
            whole = "plan=fixed pieces_per_row=1 " in d and " workspace=0" in d
            assert whole != cut, (longest, window, total, d)


def test_mla_little_work_runs_a_wave_per_tile(pkg, monkeypatch):
    """16 heads always; more heads, a workgroup per 16 of them, where the rounds of 64 tokens per CU are few.  A call that brings the room of the
    plan that stood there before keeps it, and the switch turns it off."""
    takes = lambda Hq, S, longest, **kw: "a wave per tile" in pkg._lib.describe_mla_plan(
        _mla_params(pkg, Hq, S=S, T=S, max_kv=longest, sum_kv=S * longest * 3 // 4, **kw), False)
    assert takes(16, 64, 16384) and takes(16, 1, 40, P=1, fp8=True) and takes(5, 300, 3000) and not takes(16, 64, 16384, soft_cap=30.0)
    assert takes(32, 64, 16384, fp8=True) and not takes(32, 64, 16384) and takes(24, 8, 1500)
    assert takes(64, 20, 1000) and not takes(64, 40, 4000) and takes(64, 10, 4000, fp8=True) and takes(64, 30, 2000, P=16)
    assert takes(128, 3, 4000) and takes(128, 16, 1000, fp8=True) and not takes(128, 64, 1000) and not takes(160, 1, 100)
    # both sides of the limits, in tokens of the rows; whole rows of e4m3, pieces of 512 of long bf16 rows
    def sums(Hq, S, longest, tokens, **kw):
        return "a wave per tile" in pkg._lib.describe_mla_plan(_mla_params(pkg, Hq, S=S, T=S, max_kv=longest, sum_kv=tokens, **kw), False)

    assert not sums(16, 3, 8000, 16383, fp8=True) and sums(16, 3, 8000, 16384, fp8=True) and sums(16, 3, 8000, 16383, fp8=True, P=16)
    assert sums(16, 5, 256, 700, fp8=True) and not sums(16, 5, 257, 700, fp8=True) and sums(16, 1, 600, 500)
    for rounds, waves in ((4.9, True), (5, False), (14.9, False), (15, True)):
        assert sums(32, 20, 9000, int(rounds * 8192), fp8=True) == waves and sums(32, 20, 9000, int(rounds * 8192), fp8=True, P=16), rounds
    for P, limit in ((64, 9), (16, 22)):
        assert sums(64, 20, 9000, limit * 4096 - 1, fp8=True, P=P) and not sums(64, 20, 9000, limit * 4096, fp8=True, P=P)
    assert not sums(16, 31, 2200, 40000) and sums(16, 31, 1000, 20000) and sums(16, 31, 2200, 40000, P=16) and sums(16, 31, 2200, 40000, fp8=True)
    assert not sums(32, 3, 12200, 18000) and sums(32, 6, 4800, 22000)
    p = _mla_params(pkg, 16, S=20, T=20, max_kv=1500, sum_kv=18000)
    assert "plan=fixed pieces_per_row=12" in pkg._lib.describe_mla_plan(p, False)  # one round of pieces of 128 tokens
    monkeypatch.setenv("RPA_MLA_WAVES", "0")
    assert not takes(16, 64, 16384)


@pytest.mark.parametrize("Hq", [112, 128, 129, 144, 160, 256])
def test_mla_more_than_128_heads_never_run_a_wave_per_tile(pkg, monkeypatch, Hq):
    """A share of the balanced plan has room for partial rows of 128 heads: the switch sends no more than that to the kernel of a wave per tile, on
    either plan, for rows of sequences and of tokens."""
    monkeypatch.setenv("RPA_MLA_WAVES", "1")
    for S, longest, fp8 in ((20, 16000, False), (1, 100, False), (300, 3000, True)):
        for token_rows in (False, True):
            d = pkg._lib.describe_mla_plan(_mla_params(pkg, Hq, S=S, T=S, max_kv=longest, sum_kv=S * longest * 3 // 4, fp8=fp8), token_rows)
            assert ("a wave per tile" in d) == (Hq <= 128), d


def test_mla_chunks_of_few_tokens_run_a_wave_per_tile(pkg, monkeypatch):
    """Chunk tokens that could share workgroups: a wave per tile and whole rows up to some rounds of the CUs, groups beyond, with windows and where the
    switch says so.  Short whole rows of more heads: by the workgroups too."""
    def plan(Hq, T, longest, S=2, rows=True, **kw):
        return pkg._lib.describe_mla_plan(_mla_params(pkg, Hq, S=S, T=T, max_kv=longest, sum_kv=T * longest * 3 // 4, **kw), rows)

    for Hq, most, kw in ((16, 512, {}), (32, 256, {}), (64, 128, {}), (16, 640, dict(fp8=True)), (32, 320, dict(fp8=True)), (16, 1024, dict(fp8=True, P=16)),
                         (32, 384, dict(fp8=True, P=16))):
        for T, waves in ((most, True), (most + 1, False)):
            d = plan(Hq, T, 250, **kw)
            assert ("a wave per tile" in d) == waves and ("token_groups=off" in d) == waves and "pieces_per_row=1 " in d and " workspace=0" in d, (Hq, T, kw, d)
    assert "token_groups=off" not in plan(16, 300, 4000, window=1000) and "a wave per tile" in plan(16, 300, 4000)
    for T, waves in ((170, True), (171, False)):  # heads that form no groups: up to two rounds of workgroups
        assert ("a wave per tile" in plan(40, T, 340, fp8=True, P=16)) == waves, T
    p = _mla_params(pkg, 16, S=1, T=137, max_kv=4610, sum_kv=137 * 4542)  # rows of nearly one length: no tail in a round of its own
    assert "pieces_per_row=1 " in pkg._lib.describe_mla_plan(p, True)
    for Hq, S, longest, waves, kw in ((128, 48, 100, True, {}), (128, 49, 100, False, {}), (128, 64, 100, True, dict(fp8=True)), (128, 65, 100, False, dict(fp8=True)),
                                      (64, 48, 200, True, {}), (64, 49, 200, False, {}), (32, 96, 200, True, {}), (32, 97, 200, False, {}), (16, 256, 200, True, {})):
        assert ("a wave per tile" in plan(Hq, S, longest, S=S, rows=False, **kw)) == waves, (Hq, S, kw)
    for tokens, kw, waves in ((245759, {}, False), (245760, {}, True), (200000, dict(fp8=True), True), (200000, dict(P=16), True)):  # long ragged rows
        p = _mla_params(pkg, 16, S=20, T=20, max_kv=16000, sum_kv=tokens, **kw)
        assert ("a wave per tile" in pkg._lib.describe_mla_plan(p, False)) == waves, (tokens, kw)
    monkeypatch.setenv("RPA_MLA_WAVES", "0")
    assert "token_groups=wide" in plan(16, 100, 250)


def test_mla_chunk_tokens_are_counted_as_rows(pkg):
    """Lengths on the host and no sum from the caller: the operator adds up what every query token sees, which is what the plans go by.  With the
    sequences' lengths in its place 2048 tokens on 4096 would run eight sibling workgroups each, 300 on 1000 in sixteen pieces."""
    total = pkg.mla._host_visible_sum
    rng = np.random.default_rng(3)
    q, old = rng.integers(0, 40, 9), rng.integers(0, 300, 9)
    cu, kv = np.concatenate([[0], np.cumsum(q)]).astype(np.int32), (q + old).astype(np.int32)
    want = sum(int(o) + j + 1 for n, o in zip(q[:7], old) for j in range(n))
    assert total(kv, cu, 7, False) == want and total(torch.from_numpy(kv), torch.from_numpy(cu), 7, False) == want
    assert total(kv, cu, 7, True) == int(kv[:7].sum()) and total(kv, None, 7, False) == 0 and total(None, cu, 7, False) == 0
    for n, each, kv_len, fp8, P in ((4, 512, 4608, True, 64), (4, 512, 4608, False, 16), (1, 300, 1300, False, 64)):
        kv, cu = np.full(n, kv_len, np.int32), np.arange(n + 1, dtype=np.int32) * each
        p = _mla_params(pkg, 128, P=P, fp8=fp8, S=n, T=n * each, max_kv=kv_len, sum_kv=total(kv, cu, n, False))
        d = pkg._lib.describe_mla_plan(p, True)
        assert "a wave per tile" not in d and "pieces_per_row=1 " in d and " workspace=0" in d, d


def test_mla_chunk_tokens_are_cut_by_the_longest(pkg, monkeypatch):
    """Tokens of chunks, mostly as long as the longest: pieces that one round of workgroups holds, none of short rows of many; emptier ones by the mean."""
    def pieces(Hq, T, longest, percent, **kw):
        d = pkg._lib.describe_mla_plan(_mla_params(pkg, Hq, S=2, T=T, max_kv=longest, sum_kv=-(-T * longest * percent // 100), **kw), True)
        return int(d.split("pieces_per_row=")[1].split()[0])

    for T in (40, 100, 127, 128, 129, 200):
        assert pieces(128, T, 4000, 70) == max(1, 256 // T), T
    assert pieces(128, 160, 4000, 65) == 1 and pieces(128, 160, 4000, 64) > 1 and pieces(128, 90, 4000, 69) > 2
    for longest, f8, cut in ((512, False, False), (513, False, True), (384, True, False), (385, True, True)):
        assert (pieces(128, 65, longest, 50, fp8=f8) > 1) == cut, (longest, f8)
    assert pieces(64, 65, 512, 50, fp8=True) == 1 and pieces(128, 64, 512, 70) > 1
    monkeypatch.setenv("RPA_MLA_MIN_CHUNK", "32")  # shorter pieces asked for
    assert pieces(128, 65, 512, 70) > 1


def test_mla_pages_that_the_wide_loops_do_not_take(pkg):
    """The wide loops: bytes inside a page in 32 bits, masks in front of a scale that has to be positive."""
    d = pkg._lib.describe_mla_plan
    for P, name in ((16, "wide loop of pages of 16"), (64, "shape=mla_wide")):
        p = _mla_params(pkg, 128, P=P)
        assert name in d(p, False)
        for scale in (-0.07, 0.0, 1e-30, float("nan")):
            p.sm_scale = scale
            assert name not in d(p, False), scale
        p.sm_scale = 0.07
        for stride, wide in ((2**31 // P - 8, True), (2**31 // P, False), (2**31 // P + 576, False)):
            p.row_stride = stride
            assert (name in d(p, False)) == wide, (P, stride)


def test_mla_shape_table_rows(pkg, monkeypatch):
    def params(Hq, P=64, fp8=False, S=64, T=64, max_kv=16384, sum_kv=590000, soft_cap=0.0):
        p = pkg._lib.RpaMlaParams()
        for f in ("ql_nope", "q_pe", "out", "cache_kv", "kv_lens", "page_indices", "cu_q_lens", "cu_kv_lens"):
            setattr(p, f, 0x1000)
        p.num_tokens, p.num_seqs, p.num_q_heads = T, S, Hq
        p.lkv_dim, p.rope_dim, p.page_size, p.total_pages = 512, 64, P, 1 << 16
        p.row_stride, p.rope_offset = 576, 512
        p.max_kv_len, p.sum_kv_len, p.sm_scale, p.soft_cap = max_kv, sum_kv, 0.07, soft_cap
        p.cache_dtype = pkg._lib.RPA_KV_FP8_E4M3 if fp8 else pkg._lib.RPA_KV_BF16
        return p

    d = pkg._lib.describe_mla_plan
    c5 = d(params(128), False)
    assert "shape=mla_wide" in c5 and "waves_per_wg=4" in c5 and "plan=balanced" in c5 and "workgroups=256" in c5
    assert "shape=mla_pipe" in d(params(128, fp8=True), False)
    ragged = params(16, S=20, T=20, max_kv=16000, sum_kv=200000)
    assert "shape=mla_shared_16" in d(ragged, False) and "share=4" in d(ragged, False)
    for Hq, plan in ((16, "balanced"), (128, "fixed")):  # a wave per tile: four waves, 16 heads
        text = d(params(16) if Hq == 16 else params(128, S=1, T=1, max_kv=500, sum_kv=500), False)
        assert "shape=mla_waves" in text and " waves_per_wg=4 heads_per_wg=16 share=1 " in text and f"plan={plan}" in text, text
    assert "shape=mla_shared_64" in d(params(48), False)
    assert "shape=mla_compiled" in d(params(128, P=16), False)
    assert "shape=mla_compiled" in d(params(128, soft_cap=30.0), False)
    assert "shape=mla_compiled" in d(params(160), False)
    # query tokens of a chunk with few heads share a workgroup: on the wide loop for bf16 latents without a window
    chunk = dict(S=4, T=4096, max_kv=8192, sum_kv=20000)
    assert "token_groups=off" in d(params(16), False) and "token_groups=off" in d(params(16), True)  # decode rows
    assert "token_groups=wide" in d(params(16, **chunk), True) and "waves_per_wg=4" in d(params(16, **chunk), True)
    assert "token_groups=eight_waves " in d(params(32, fp8=True, **chunk), True)
    windowed = params(64, **chunk)
    windowed.sliding_window = 512
    assert "token_groups=eight_waves " in d(windowed, True)
    assert "token_groups=off" in d(params(48, **chunk), True) and "token_groups=off" in d(params(128, **chunk), True)
    monkeypatch.setenv("RPA_MLA_TOKEN_GROUPS", "0")
    assert "token_groups=off" in d(params(16, **chunk), True)
    monkeypatch.delenv("RPA_MLA_TOKEN_GROUPS")
    monkeypatch.setenv("RPA_MLA_WIDE", "0")
    assert "token_groups=eight_waves " in d(params(16, **chunk), True)
    assert "shape=mla_pipe" in d(params(128), False)
    monkeypatch.setenv("RPA_MLA_PIPE", "0")
    assert "shape=mla_compiled" in d(params(128), False)
    assert "token_groups=eight_waves_compiled" in d(params(16, **chunk), True)
