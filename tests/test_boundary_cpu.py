"""CPU-side checks of the drop-in boundary: the C-ABI library loads and exports every entry
point include/zenyx_kv.h declares, argument errors come back as status codes (no GPU
needed: validation precedes every HIP call), and the host-side logic (ring access
sequence, tiering sizes, reference timeline) matches the oracle and closed forms."""
import ctypes
import os
import re
import subprocess
import sys

import numpy as np
import pytest

from oracle import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def header_symbols():
    text = open(os.path.join(ROOT, "include", "zenyx_kv.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(zx_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_header_symbol():
    from zenyx_amd import _native

    lib = _native.load()
    syms = header_symbols()
    assert len(syms) >= 15
    for s in syms:
        assert hasattr(lib, s), f"libzenyx_kv.so does not export {s}"
        assert s in _native.SIGNATURES, f"{s} has no ctypes signature"
    assert lib.zx_abi_version() == _native.ABI_VERSION


def test_argument_errors_are_status_codes():
    from zenyx_amd import _native as N

    lib = N.load()
    rc = lib.zx_kv_gather_dequant(None, 10, 8, 128, 16, None, None, 4, None, 2, 64, None, None, None, None)
    assert rc == N.ZX_ERR_INVALID and b"null pointer" in lib.zx_last_error()
    rc = lib.zx_kv_gather_dequant(ctypes.c_void_p(16), 10, 8, 96, 16, ctypes.c_void_p(16), ctypes.c_void_p(16), 4,
                                  ctypes.c_void_p(16), 2, 64, ctypes.c_void_p(16), ctypes.c_void_p(16), None, None)
    assert rc == N.ZX_ERR_UNSUPPORTED and b"head_dim" in lib.zx_last_error()
    # bulk arrays off a 16-byte boundary are refused before any device call
    p16, p8 = ctypes.c_void_p(16), ctypes.c_void_p(24)
    rc = lib.zx_kv_gather_dequant(p8, 10, 8, 128, 16, p16, p16, 4, p16, 2, 64, p16, p16, None, None)
    assert rc == N.ZX_ERR_INVALID and b"16-byte aligned" in lib.zx_last_error()
    rc = lib.zx_kv_quant_append(p8, 16 * 2 * 8 * 128, 1, 16, 8, 128, p16, None, 1, p16, 1, 16, p16,
                                2 * 8 * 16 * 128, 1, p16, 0, None, p16, 1 << 20, None)
    assert rc == N.ZX_ERR_INVALID and b"16-byte aligned" in lib.zx_last_error()
    rc = lib.zx_int8_legacy_quant(ctypes.c_void_p(16), 0, 0, ctypes.c_void_p(16), ctypes.c_void_p(16),
                                  ctypes.c_void_p(16), 256, None)
    assert rc == N.ZX_ERR_INVALID and b"empty" in lib.zx_last_error()
    rc = lib.zx_belady_simulate(None, None, None, 10, 0, 10, 5, 0, ctypes.c_void_p(16), ctypes.c_void_p(16),
                                ctypes.c_void_p(16), None, None, 0, None, None, 0, None)
    assert rc == N.ZX_ERR_INVALID and b"capacity" in lib.zx_last_error()
    with pytest.raises(ValueError):
        N.check(N.ZX_ERR_INVALID, "x")
    with pytest.raises(N.ZenyxNativeError):
        N.check(N.ZX_ERR_HIP, "x")


def test_workspace_queries_are_host_only():
    from zenyx_amd import _native as N

    lib = N.load()
    assert lib.zx_kv_quant_append_workspace_bytes(32, 74902, 8, 128) >= 74902 * 8
    assert lib.zx_belady_simulate_workspace_bytes(20_971_520, 1_310_720) >= (20_971_520 + 1_310_720) // 8
    assert lib.zx_belady_argmax_workspace_bytes(1000) >= 16


def test_decode_workspace_of_unsupported_head_dims():
    """The wrapper asks for the size before the call is checked: for a head_dim no kernel takes
    the answer is 0, and the call itself is refused.  In a process of its own: a division by
    zero here would end it."""
    code = """
import ctypes
from zenyx_amd import _native as N
lib, p = N.load(), ctypes.c_void_p(16)
for d in (-8, 0, 1, 8, 15, 96, 512, 4096, 8192, 1 << 20):
    assert lib.zx_paged_attention_decode_workspace_bytes(1, 8, 8, d, 4, 16) == 0, d
    rc = lib.zx_paged_attention_decode(p, 8, p, 4, 8, d, 16, p, p, 4, p, 1, 0.1, p, None, p, 1 << 20, None)
    assert rc == N.ZX_ERR_UNSUPPORTED and b"head_dim" in lib.zx_last_error(), (d, rc)
for d in (64, 128, 256):
    assert lib.zx_paged_attention_decode_workspace_bytes(1, 8, 8, d, 4, 16) > 0
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.returncode, r.stderr[-2000:])


@pytest.mark.parametrize("L,R,S", [(1, 1, 5), (3, 8, 4), (2, 4, 7)])
def test_ring_access_sequence_sizes(L, R, S):
    """The trace itself is built on the GPU (tests/test_gpu_dropin.py); here its sizes, and
    the oracle's trace against the closed form of ring step r, device d -> shard (d - r) mod R."""
    from zenyx_amd.train.belayd_kv_cache_tiering import RingAttentionAccessSequence

    seq = RingAttentionAccessSequence(L, R, S)
    tr = O.ring_trace(L, R, S)
    assert len(seq) == tr.size and seq.n_pages == L * R * S
    fwd = np.array([(l * R + (d - r) % R) * S + i for l in range(L) for r in range(R) for d in range(R)
                    for i in range(S)], np.int32)
    np.testing.assert_array_equal(tr, np.concatenate([fwd, fwd[::-1]]))


def test_tiering_manager_sizes_at_baseline_config():
    from zenyx_amd.train.belayd_kv_cache_tiering import BeladyKVCacheTieringManager

    m = BeladyKVCacheTieringManager(num_devices=8, context_length=2**20, num_layers=80, num_kv_heads=8,
                                    head_dim=128, page_tokens=64, hbm_budget_bytes=64e9)
    assert m.page_bytes == 128 * 1024
    assert m.pages_per_shard == 2048
    assert m.n_pages == 1_310_720
    assert m.capacity == 488_281
    assert len(m.sequence) == 20_971_520
    # the README constructor (README.md:93-97)
    r = BeladyKVCacheTieringManager(num_devices=8, context_length=4096, num_layers=12)
    assert r.capacity == r.n_pages == 12 * 8 * 8


def test_build_ring_timeline_matches_reference():
    from zenyx_amd.streaming import build_ring_timeline

    for n in (1, 2, 7):
        assert build_ring_timeline(n) == O.ref_ring_timeline(n)


def header_constants():
    """NAME -> value of every ZX_* constant the header defines (enum members and #defines)."""
    text = open(os.path.join(ROOT, "include", "zenyx_kv.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    consts = {}
    for name, val in re.findall(r"\b(ZX_[A-Z0-9_]+)\s*=\s*(-?\d+)", text):
        consts[name] = int(val)
    for name, val, sh in re.findall(r"#define\s+(ZX_[A-Z0-9_]+)\s+\(?(\d+)u?\s*(?:<<\s*(\d+))?", text):
        consts[name] = int(val) << int(sh or 0)
    return consts


def test_header_constants_match_the_python_binding():
    from zenyx_amd import _native as N

    consts = header_constants()
    for name in ("ZX_PREFILL_MERGE", "ZX_PREFILL_INIT", "ZX_PREFILL_BF16", "ZX_PREFILL_FAST_P", "ZX_PREFILL_EXACT_P",
                 "ZX_PREFILL_LAST", "ZX_PREFILL_FINAL",
                 "ZX_HEADS_TWO_PASS", "ZX_HEADS_SINGLE_PASS", "ZX_APPEND_STATIC_SCALES", "ZX_APPEND_SATURATE",
                 "ZX_APPEND_TWO_PASS", "ZX_KERR_PAGE_RANGE", "ZX_KERR_POS_RANGE", "ZX_KERR_SPIN", "ZX_KERR_OVERFLOW",
                 "ZX_ERR_INVALID", "ZX_ERR_UNSUPPORTED", "ZX_ERR_WORKSPACE"):
        assert name in consts, f"{name} not found in the header"
        assert getattr(N, name) == consts[name], f"{name}: header {consts[name]}, binding {getattr(N, name)}"


def test_exclusive_flags_are_refused_before_any_device_call():
    from zenyx_amd import _native as N

    lib = N.load()
    p = ctypes.c_void_p(16)
    rc = lib.zx_fp8_quant_heads(p, 1, 1, 1, 16, p, p, N.ZX_HEADS_TWO_PASS | N.ZX_HEADS_SINGLE_PASS, None, None, 0,
                                None)
    assert rc == N.ZX_ERR_INVALID and b"together" in lib.zx_last_error()
    rc = lib.zx_fp8_quant_heads(p, 1, 1, 1, 16, p, p, 64, None, None, 0, None)
    assert rc == N.ZX_ERR_INVALID and b"unknown flag" in lib.zx_last_error()
    for fl, msg in ((N.ZX_APPEND_TWO_PASS | N.ZX_APPEND_SINGLE_PASS, b"together"), (64, b"unknown flag")):
        rc = lib.zx_kv_quant_append(p, 16 * 2 * 8 * 128, 1, 16, 8, 128, p, None, 1, p, 1, 16, p, 2 * 8 * 16 * 128, 1,
                                    p, fl, None, None, 0, None)
        assert rc == N.ZX_ERR_INVALID and msg in lib.zx_last_error()
    for fn, extra in ((lib.zx_paged_attention_prefill, ()), (lib.zx_paged_attention_ring, (1,))):
        args = [p, 16, p, p, 8, p, 10, 2, 128, 16, p, p, 4] + [p, p] + list(extra) + [1, 16, 1, 0.1]
        rc = fn(*args, N.ZX_PREFILL_BF16 | N.ZX_PREFILL_FAST_P | N.ZX_PREFILL_EXACT_P, None, None, p, None, None)
        assert rc == N.ZX_ERR_INVALID and b"together" in lib.zx_last_error()
        rc = fn(*args, N.ZX_PREFILL_BF16 | N.ZX_PREFILL_LAST, None, None, p, None, None)
        assert rc == N.ZX_ERR_INVALID and b"ZX_PREFILL_LAST needs" in lib.zx_last_error()
        rc = fn(*args, N.ZX_PREFILL_BF16 | N.ZX_PREFILL_FINAL, None, None, p, None, None)
        assert rc == N.ZX_ERR_INVALID and b"ZX_PREFILL_FINAL needs" in lib.zx_last_error()
        rc = fn(*args, 128 | N.ZX_PREFILL_BF16, None, None, p, None, None)
        assert rc == N.ZX_ERR_INVALID and b"unknown flags" in lib.zx_last_error()
    # FINAL on a non-causal step
    args = [p, 16, p, p, 8, p, 10, 2, 128, 16, p, p, 4, p, p, 1, 16, 0, 0.1]
    rc = lib.zx_paged_attention_prefill(*args, N.ZX_PREFILL_MERGE | N.ZX_PREFILL_BF16 | N.ZX_PREFILL_FINAL, p, p, p,
                                        None, None)
    assert rc == N.ZX_ERR_INVALID and b"ZX_PREFILL_FINAL needs" in lib.zx_last_error()


def test_attention_precision_names():
    import torch

    from zenyx_amd import kv

    assert kv.PRECISIONS == ("f16", "bf16", "exact")
    t = torch.zeros(1)
    with pytest.raises(ValueError, match="precision"):
        kv.ring_attention_fp8(t, t, t, t, t, t, t, ring_degree=1, precision="fp8")
    with pytest.raises(ValueError, match="precision"):
        kv.paged_attention_prefill(t, t, t, t, t, t, t, t, precision="half")


def test_stream_of_every_way_to_name_a_device(monkeypatch):
    """A torch.device with an index takes the short way; a text, a number, no index and None
    are left to torch, as it names devices."""
    import torch

    from zenyx_amd import _native as N

    class Stream:
        cuda_stream = 77

    asked = []
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: asked.append(d) or Stream())
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda i: 1000 + i, raising=False)
    assert N.stream_ptr(torch.device("cuda", 3)) == 1003 and asked == []
    others = ["cuda", "cuda:0", 1, torch.device("cuda"), None]
    assert [N.stream_ptr(d) for d in others] == [77] * 5 and asked == others


@pytest.mark.parametrize("single_launch", [True, False])
@pytest.mark.parametrize("form", ["int32", "int64", "row", "strided", "row_int64"])
def test_ring_shard_bounds_of_every_kv_len(monkeypatch, form, single_launch):
    """ring_attention_fp8 hands shard r the keys [floor(n r / R), floor(n (r + 1) / R)) whatever
    the dtype, strides or leading dimensions of 1 of kv_len (on the CPU: by torch)."""
    import torch

    from zenyx_amd import kv

    lens, R = torch.tensor([0, 5, 8191, 2**31 - 1, 17], dtype=torch.int32), 3
    kv_len = {"int32": lens, "int64": lens.long(), "row": lens[None], "row_int64": lens.long()[None],
              "strided": torch.stack([lens, lens], 1)[:, 0]}[form]
    got = []
    monkeypatch.setattr(kv, "paged_attention_ring", lambda q, cu, qp, pool, sc, bt, kb, ke, **_: got.extend(
        zip(kb.tolist(), ke.tolist())))
    monkeypatch.setattr(kv, "paged_attention_prefill", lambda q, cu, qp, pool, sc, bt, kb, ke, **_: got.append(
        (kb.tolist(), ke.tolist())))
    q = torch.zeros((1, 1, 128), dtype=torch.bfloat16)
    kv.ring_attention_fp8(q, None, None, None, None, None, kv_len, R, max_q_per_seq=1, single_launch=single_launch)
    n = lens.tolist()
    assert got == [([x * r // R for x in n], [x * (r + 1) // R for x in n]) for r in range(R)]


def test_prefill_plan_under_a_loose_bound():
    """max_q_per_seq is a bound: one far above the call's rows gives the same plan (the same
    workspace) as the number of its rows."""
    from zenyx_amd import _native as N

    size = N.load().zx_paged_attention_ring_workspace_bytes
    for n_q, n_seqs, Hq, Hkv in ((64, 1, 32, 8), (256, 4, 32, 8), (33, 3, 8, 8), (700, 2, 16, 8)):
        tight = size(n_q, Hq, Hkv, 16, 600, n_seqs, n_q, 1, N.ZX_PREFILL_BF16)
        assert tight > 0
        for most in (n_q + 1, 131072, 2**31 - 1):
            assert size(n_q, Hq, Hkv, 16, 600, n_seqs, most, 1, N.ZX_PREFILL_BF16) == tight


def test_prefill_is_not_cut_where_its_tiles_fill_the_chip():
    """Two parts a tile only cost where the uncut tiles take one full round of blocks (two per
    CU; 256 CUs where there is no device)."""
    from zenyx_amd import _native as N

    size = N.load().zx_paged_attention_ring_workspace_bytes
    cus = 256
    try:
        import torch
        if torch.cuda.is_available():
            cus = torch.cuda.get_device_properties(0).multi_processor_count
    except RuntimeError:
        pass
    tiles = 2 * cus // 8  # sequences of one tile for 8 head groups
    for n_seqs, cut in ((tiles, False), (tiles * 15 // 16, False), (tiles * 3 // 4, True), (tiles // 4, True)):
        assert (size(32 * n_seqs, 32, 8, 16, 512, n_seqs, 32, 1, N.ZX_PREFILL_BF16) > 0) == cut, n_seqs
