"""Blocks of queries over the FP8 pages (one ring step of QuantizedRingAttention,
README.md:344) and ring attention composed from such steps on one GPU, against the C
oracle (itself pinned against torch float64 in test_oracle.py).

Tolerance: the kernel computes scores in fp32 on matrix cores (bf16 q, K codes exact in
bf16) and an exp2-domain online softmax; how P enters P.V sets the bound per output
channel (the row sums use the same P, so a row is an average of V under weights
perturbed by at most e relative, which moves it by at most 2 e max|V|):
  "f16"   (default, P x 2^7 fp16): one bf16 ulp of the exact value + 2^-10 max|V| (e = 2^-11);
  "bf16"  (P rounded to bf16):     one ulp + 2^-7 max|V|  (e = 2^-8);
  "exact" (P as bf16 hi + lo):     e = 2^-16, a worst case of one ulp + 2^-15 max|V|; the
                                   rounding errors are independent and average out, and
                                   the tests hold this mode to one ulp + 2^-17 max|V|;
the oracle value, rounded to bf16, stands for the exact one: one more ulp for the modes
whose bound is not far below an ulp.  lse2 (log2 of the softmax denominator) within 2e-5
(absolute + relative), plus log2 of the weights' perturbation, e / ln 2, for "f16" and
"bf16" (the denominator is the sum of the same rounded weights, which keeps ring steps
merged by lse2 an average under those weights).
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from zenyx_amd import kv
from test_gpu_attention import assert_within_bound, bf16_to_f32, kernels_of, least_us

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def bits16(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def make(Hq, Hkv, P, n_q, q_pos0, kv_len, seed, n_pages=None):
    rng = np.random.default_rng(seed)
    D = 128
    B = len(n_q)
    max_blocks = max(1, -(-max(kv_len) // P))
    n_pages = n_pages or B * max_blocks + 3
    pool = rng.integers(0, 256, (n_pages, 2, Hkv, P, D), dtype=np.uint8)
    pool[(pool & 0x7F) == 0x7F] = 0x3A
    perm = rng.permutation(n_pages)
    bt = perm[:B * max_blocks].reshape(B, max_blocks).astype(np.int32)
    scales = rng.uniform(1e-3, 0.05, (2, Hkv)).astype(np.float32)
    cu = np.concatenate([[0], np.cumsum(n_q)]).astype(np.int32)
    q = torch.from_numpy(rng.standard_normal((int(cu[-1]), Hq, D)).astype(np.float32)).to(torch.bfloat16)
    return q, pool, scales, bt, cu, np.asarray(q_pos0, np.int32)


def vmax_rows(pool, scales, bt, cu, kv_begin, kv_end, Hq):
    """Per (row, query head, channel): max |V| over the sequence's key range (a bound
    for the keys the row actually uses)."""
    dec = np.abs(O.e4m3_decode(np.arange(256, dtype=np.uint8)).astype(np.float64))
    n_pages, _, Hkv, P, D = pool.shape
    out = np.zeros((int(cu[-1]), Hq, D))
    for b in range(len(cu) - 1):
        t = np.arange(kv_begin[b], kv_end[b])
        if t.size == 0:
            continue
        pages = bt[b, t // P]
        for hq in range(Hq):
            h = hq // (Hq // Hkv)
            out[cu[b]:cu[b + 1], hq] = np.nanmax(dec[pool[pages, 1, h, t % P, :]], axis=0) * abs(float(scales[1, h]))
    return out


P_BOUND = {"exact": (1, 2.0 ** -17), "f16": (2, 2.0 ** -10), "bf16": (2, 2.0 ** -7)}  # (ulps, bound on |V|)
LSE_EXTRA = {"exact": 0.0, "f16": 2.0 ** -11 / np.log(2.0), "bf16": 2.0 ** -8 / np.log(2.0)}


def assert_precision(got_bits, want_bits, vmax, precision="f16"):
    ulps, e = P_BOUND[precision]
    return assert_within_bound(got_bits, want_bits, vmax, e, ulps)


def run_step(q, pool, scales, bt, cu, q_pos0, kb, ke, causal, precision="f16"):
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    o_acc = torch.empty(q.shape, dtype=torch.float32, device=DEV)
    lse = torch.empty(q.shape[:2], dtype=torch.float32, device=DEV)
    out = kv.paged_attention_prefill(q.to(DEV), t(cu), t(q_pos0), t(pool), t(scales), t(bt), t(kb), t(ke),
                                     causal=causal, o_acc=o_acc, lse2=lse, first=True, check=True,
                                     precision=precision)
    return out, lse


CASES = [  # Hq, Hkv, P, n_q, q_pos0, kv_begin, kv_end
    (8, 2, 16, [37, 5, 64], [0, 20, 100], [0, 3, 17], [37, 25, 164]),
    (32, 8, 16, [130, 1], [500, 0], [0, 0], [630, 1]),
    (4, 4, 32, [70, 33], [0, 64], [5, 70], [70, 70]),       # second: empty key range
    (6, 3, 16, [20, 0, 45], [10, 0, 5], [0, 0, 0], [30, 0, 50]),  # a sequence with no queries
    (2, 1, 48, [129], [300], [40], [429]),
]


@pytest.mark.parametrize("precision", ["f16", "exact", "bf16"])
@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("causal", [True, False])
def test_prefill_step_matches_oracle(case, causal, precision):
    Hq, Hkv, P, n_q, q_pos0, kb, ke = CASES[case]
    print(f"prefill step case {case} causal={causal} precision={precision}", flush=True)
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, n_q, q_pos0, ke, seed=case)
    kb, ke = np.asarray(kb, np.int32), np.asarray(ke, np.int32)
    out, lse = run_step(q, pool, scales, bt, cu, qp, kb, ke, causal, precision)
    torch.cuda.synchronize()
    sm = float(np.float32(1.0 / np.sqrt(128)))
    want, wlse, err = O.paged_attention_prefill(bits16(q), cu, qp, pool, scales, bt, kb, ke, causal, sm)
    assert err == 0
    assert_precision(bits16(out), want, vmax_rows(pool, scales, bt, cu, kb, ke, Hq), precision)
    g = lse.cpu().numpy()
    fin = np.isfinite(wlse)
    np.testing.assert_array_equal(np.isfinite(g), fin)
    assert np.all(np.abs(g[fin] - wlse[fin]) <= 2e-5 * (1 + np.abs(wlse[fin])) + LSE_EXTRA[precision])


_RING_CASE = {}


def _ring_case():
    """One set of inputs and its oracle result, shared by the ring degrees."""
    if not _RING_CASE:
        Hq, Hkv, P = 32, 8, 16
        n_q, lens, q_pos0 = [256, 77, 512], [256, 300, 1024], [0, 223, 512]  # queries end at the last key
        q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, n_q, q_pos0, lens, seed=41)
        zeros, lens_a = np.zeros(len(lens), np.int32), np.asarray(lens, np.int32)
        sm = float(np.float32(1.0 / np.sqrt(128)))
        want, _, err = O.paged_attention_prefill(bits16(q), cu, qp, pool, scales, bt, zeros, lens_a, True, sm)
        assert err == 0
        _RING_CASE.update(q=q, pool=pool, scales=scales, bt=bt, cu=cu, qp=qp, lens=lens_a, want=want,
                          vmax=vmax_rows(pool, scales, bt, cu, zeros, lens_a, Hq))
    return _RING_CASE


@pytest.mark.parametrize("precision", ["f16", "exact"])
@pytest.mark.parametrize("single_launch", [True, False])
@pytest.mark.parametrize("ring", [1, 3, 8, 70])  # 70: more ranges than a block keeps in LDS
def test_ring_attention_equals_full_attention(ring, single_launch, precision):
    c = _ring_case()
    print(f"ring {ring} single_launch={single_launch} precision={precision}", flush=True)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    out = kv.ring_attention_fp8(c["q"].to(DEV), t(c["cu"]), t(c["qp"]), t(c["pool"]), t(c["scales"]), t(c["bt"]),
                                t(c["lens"]), ring_degree=ring, causal=True, check=True, single_launch=single_launch,
                                precision=precision)
    torch.cuda.synchronize()
    worst = assert_precision(bits16(out), c["want"], c["vmax"], precision)
    print(f"  worst |err| / max|V| = {worst:.3g}", flush=True)


@pytest.mark.parametrize("precision", ["f16", "exact"])
def test_last_step_leaves_the_running_output(precision):
    """ZX_PREFILL_LAST: the last step of a ring writes the same bf16 rows as a merging
    step and leaves o_acc / lse2 as they were."""
    c = _ring_case()
    print(f"last step precision={precision}", flush=True)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    q, cu, qp, pool, scales, bt = c["q"].to(DEV), t(c["cu"]), t(c["qp"]), t(c["pool"]), t(c["scales"]), t(c["bt"])
    lens = c["lens"].astype(np.int64)
    R = 3
    bounds = [t((lens * r // R).astype(np.int32)) for r in range(R + 1)]
    o_acc = torch.empty(q.shape, dtype=torch.float32, device=DEV)
    lse2 = torch.empty(q.shape[:2], dtype=torch.float32, device=DEV)
    for r in range(R - 1):
        kv.paged_attention_prefill(q, cu, qp, pool, scales, bt, bounds[r], bounds[r + 1], o_acc=o_acc, lse2=lse2,
                                   first=r == 0, write_bf16=False, check=True, precision=precision)
    o_keep, l_keep = o_acc.clone(), lse2.clone()
    out_last = kv.paged_attention_prefill(q, cu, qp, pool, scales, bt, bounds[R - 1], bounds[R], o_acc=o_acc,
                                          lse2=lse2, first=False, check=True, precision=precision, last=True)
    torch.cuda.synchronize()
    assert torch.equal(o_acc.view(torch.int32), o_keep.view(torch.int32))
    assert torch.equal(lse2.view(torch.int32), l_keep.view(torch.int32))
    out_merge = kv.paged_attention_prefill(q, cu, qp, pool, scales, bt, bounds[R - 1], bounds[R], o_acc=o_acc,
                                           lse2=lse2, first=False, check=True, precision=precision)
    torch.cuda.synchronize()
    assert torch.equal(out_last.view(torch.int16), out_merge.view(torch.int16))
    assert not torch.equal(o_acc.view(torch.int32), o_keep.view(torch.int32))  # the merging step did write
    assert_precision(bits16(out_last), c["want"], c["vmax"], precision)
    with pytest.raises(ValueError):
        kv.paged_attention_prefill(q, cu, qp, pool, scales, bt, bounds[0], bounds[1], last=True)


def _steps(q, cu, qp, pool, scales, bt, lens, R, final, precision="f16"):
    """A causal ring of R launches over keys [0, lens) in ascending contiguous shards; out
    starts as a NaN pattern so that a row no step writes shows."""
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    lens = np.asarray(lens, np.int64)
    bounds = [t((lens * r // R).astype(np.int32)) for r in range(R + 1)]
    o_acc = torch.empty(q.shape, dtype=torch.float32, device=DEV)
    lse2 = torch.empty(q.shape[:2], dtype=torch.float32, device=DEV)
    out = torch.full(q.shape, 0x7FC1, dtype=torch.int16, device=DEV).view(torch.bfloat16)
    for r in range(R):
        kv.paged_attention_prefill(q, cu, qp, pool, scales, bt, bounds[r], bounds[r + 1], o_acc=o_acc, lse2=lse2,
                                   first=r == 0, out=out, write_bf16=final or r == R - 1, check=True,
                                   precision=precision, last=r == R - 1, final=final)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("shape", ["ragged", "queries_past_keys", "empty_shards"])
@pytest.mark.parametrize("R", [3, 8])
def test_final_steps_equal_the_merged_ring(shape, R):
    """ZX_PREFILL_FINAL: every step writes as bf16 the rows it completes and the last one
    converts only the rows it reaches; the output equals, bit for bit, the ring that merges
    every row into the running output and converts them all in the last step (the same
    fp32 value goes to bf16 either way), every row is written (none keeps the NaN pattern
    the output starts with), and it is within the default bound of the oracle."""
    if shape == "ragged":
        c = _ring_case()
        q, pool, scales, bt, cu, qp, lens = c["q"], c["pool"], c["scales"], c["bt"], c["cu"], c["qp"], c["lens"]
        Hq, want, vmax = 32, c["want"], c["vmax"]
    else:
        Hq, Hkv, P = 8, 2, 16
        if shape == "queries_past_keys":  # rows at positions past the last key see every key
            n_q, q_pos0, lens = [40, 70, 5], [10, 0, 30], [30, 50, 33]
        else:  # most shards empty, a sequence's only key in the last shard
            n_q, q_pos0, lens = [3, 4, 20], [0, 0, 0], [3, 1, 20]
        q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, n_q, q_pos0, lens, seed=23)
        lens = np.asarray(lens, np.int32)
        zeros = np.zeros(len(lens), np.int32)
        sm = float(np.float32(1.0 / np.sqrt(128)))
        want, _, err = O.paged_attention_prefill(bits16(q), cu, qp, pool, scales, bt, zeros, lens, True, sm)
        assert err == 0
        vmax = vmax_rows(pool, scales, bt, cu, zeros, lens, Hq)
    print(f"final steps: {shape}, R={R}", flush=True)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    args = (q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt), lens, R)
    got = _steps(*args, final=True)
    ref = _steps(*args, final=False)
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
    assert not torch.isnan(got.float()).any()
    assert_precision(bits16(got), want, vmax)
    with pytest.raises(ValueError):
        kv.paged_attention_prefill(q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt), t(np.zeros(len(lens), np.int32)),
                                   t(np.asarray(lens, np.int32)), causal=False, o_acc=torch.empty(q.shape,
                                   dtype=torch.float32, device=DEV), lse2=torch.empty(q.shape[:2],
                                   dtype=torch.float32, device=DEV), final=True)


def test_final_first_step_writes_every_row():
    """ZX_PREFILL_FINAL on a first step (INIT) whose key range starts past some rows: no
    earlier step finished those rows, so they are written too (no key: zeros), and the
    one-step ring (INIT | LAST | FINAL) equals a plain merging step bit for bit and the
    oracle within the default bound."""
    Hq, Hkv, P = 8, 2, 16
    n_q, q_pos0, kb, ke = [40, 70], [0, 0], [10, 30], [50, 60]
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, n_q, q_pos0, ke, seed=29)
    kb, ke = np.asarray(kb, np.int32), np.asarray(ke, np.int32)
    sm = float(np.float32(1.0 / np.sqrt(128)))
    want, _, err = O.paged_attention_prefill(bits16(q), cu, qp, pool, scales, bt, kb, ke, True, sm)
    assert err == 0
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    outs = []
    for final in (True, False):
        o_acc = torch.empty(q.shape, dtype=torch.float32, device=DEV)
        lse2 = torch.empty(q.shape[:2], dtype=torch.float32, device=DEV)
        out = torch.full(q.shape, 0x7FC1, dtype=torch.int16, device=DEV).view(torch.bfloat16)
        kv.paged_attention_prefill(q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt), t(kb), t(ke), o_acc=o_acc,
                                   lse2=lse2, first=True, out=out, check=True, last=final, final=final)
        torch.cuda.synchronize()
        outs.append(out)
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    assert not torch.isnan(outs[0].float()).any()
    assert_precision(bits16(outs[0]), want, vmax_rows(pool, scales, bt, cu, kb, ke, Hq))


@pytest.mark.parametrize("ring,single", [(1, True), (8, True), (3, False)])
def test_ring_attention_bf16_p(ring, single):
    """P rounded once to bf16 for P.V (ZX_PREFILL_FAST_P): within its bound of the oracle
    (one ulp + 2^-7 max|V|)."""
    c = _ring_case()
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    out = kv.ring_attention_fp8(c["q"].to(DEV), t(c["cu"]), t(c["qp"]), t(c["pool"]), t(c["scales"]), t(c["bt"]),
                                t(c["lens"]), ring_degree=ring, causal=True, check=True, single_launch=single,
                                precision="bf16")
    torch.cuda.synchronize()
    worst = assert_precision(bits16(out), c["want"], c["vmax"], "bf16")
    print(f"ring {ring} bf16 P: worst |err| / max|V| = {worst:.3g}", flush=True)


def test_f16_p_keeps_small_weights():
    """The fp16 mode on rows where one key outweighs each of the ~200 others by 2^15.5 (q all
    ones, K all ones but key 7 = 20: scores 15.5 log2 units apart): the small weights sum to
    ~2^-8 of the row and lie below fp16's normal range unless P carries its 2^7 factor, so
    losing them would miss the 2^-10 max|V| bound; within it, as the exact mode is within
    its own."""
    Hq, Hkv, P = 4, 1, 16
    _, pool, scales, bt, cu, qp = make(Hq, Hkv, P, [64], [191], [256], seed=23)
    q = torch.ones((64, Hq, 128), dtype=torch.bfloat16)
    pool[:, 0] = 0x38  # K = 1.0 (e4m3) everywhere ...
    pool[bt[0, 7 // P], 0, 0, 7 % P, :] = 0x5A  # ... but key 7 = 20.0
    scales[0, 0] = 0.05
    kb, ke = np.zeros(1, np.int32), np.full(1, 256, np.int32)
    sm = float(np.float32(1.0 / np.sqrt(128)))
    want, _, err = O.paged_attention_prefill(bits16(q), cu, qp, pool, scales, bt, kb, ke, True, sm)
    assert err == 0
    vm = vmax_rows(pool, scales, bt, cu, kb, ke, Hq)
    for precision in ("f16", "exact"):
        out, _ = run_step(q, pool, scales, bt, cu, qp, kb, ke, True, precision)
        torch.cuda.synchronize()
        worst = assert_precision(bits16(out), want, vm, precision)
        print(f"{precision}: worst |err| / max|V| = {worst:.3g}", flush=True)


@pytest.mark.parametrize("causal", [True, False])
def test_ring_ranges_in_device_order(causal):
    """zx_paged_attention_ring with the shards in the order one device of a ring of 5 sees
    them (its own shard first, then (g - r) mod 5), uneven shards, an empty shard and a
    range that starts mid-page: equal to attention over the union."""
    c = _ring_case()
    lens = c["lens"]
    R, g = 5, 3
    cuts = np.stack([np.array([0, 1, 2, 2, 4, 5]) * L // 5 for L in lens], axis=1)  # shard 2 empty
    cuts[1] = np.minimum(cuts[1] + 7, cuts[2])  # uneven: shard 0 longer, starting mid-page for shard 1
    order = [(g - r) % R for r in range(R)]
    kb = np.stack([cuts[s] for s in order]).astype(np.int32)
    ke = np.stack([cuts[s + 1] for s in order]).astype(np.int32)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    out = kv.paged_attention_ring(c["q"].to(DEV), t(c["cu"]), t(c["qp"]), t(c["pool"]), t(c["scales"]), t(c["bt"]),
                                  t(kb), t(ke), causal=causal, check=True)
    torch.cuda.synchronize()
    if causal:
        want, vmax = c["want"], c["vmax"]
    else:
        zeros = np.zeros(len(lens), np.int32)
        sm = float(np.float32(1.0 / np.sqrt(128)))
        want, _, err = O.paged_attention_prefill(bits16(c["q"]), c["cu"], c["qp"], c["pool"], c["scales"], c["bt"],
                                                 zeros, lens, False, sm)
        assert err == 0
        vmax = c["vmax"]
    assert_precision(bits16(out), want, vmax)


@pytest.mark.parametrize("precision", ["f16", "exact"])
def test_negative_scales(precision):
    """Scales of either sign (a static scale may be negative): with K's scale negative the
    scores change sign and every step takes the masked softmax path (the maximum of
    s * scale is no longer the scale times the maximum of s); V heads with a negative scale
    flip their output.  A step, causal and not, and ring attention over 3 shards in one
    launch and in separate launches."""
    Hq, Hkv, P = 8, 4, 16
    n_q, q_pos0, lens = [70, 33], [30, 0], [100, 140]
    print(f"negative scales precision={precision}", flush=True)
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, n_q, q_pos0, lens, seed=37)
    scales[0, 0::2] *= -1.0
    scales[1, 1::2] *= -1.0
    kb, ke = np.zeros(2, np.int32), np.asarray(lens, np.int32)
    sm = float(np.float32(1.0 / np.sqrt(128)))
    vm = vmax_rows(pool, scales, bt, cu, kb, ke, Hq)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    for causal in (True, False):
        want, wlse, err = O.paged_attention_prefill(bits16(q), cu, qp, pool, scales, bt, kb, ke, causal, sm)
        assert err == 0
        out, lse = run_step(q, pool, scales, bt, cu, qp, kb, ke, causal, precision)
        torch.cuda.synchronize()
        assert_precision(bits16(out), want, vm, precision)
        g = lse.cpu().numpy()
        fin = np.isfinite(wlse)
        np.testing.assert_array_equal(np.isfinite(g), fin)
        assert np.all(np.abs(g[fin] - wlse[fin]) <= 2e-5 * (1 + np.abs(wlse[fin])) + LSE_EXTRA[precision])
        for single in (False, True):
            ring = kv.ring_attention_fp8(q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt), t(ke), ring_degree=3,
                                         causal=causal, check=True, single_launch=single, precision=precision)
            torch.cuda.synchronize()
            assert_precision(bits16(ring), want, vm, precision)


def assert_nan_leak_only_in_window(got_bits, want_bits, vmax, precision, leak):
    """got equals want to the precision bound, NaN compared as a class, except that got may
    be NaN where want is not inside the boolean mask ``leak``."""
    g, w = bf16_to_f32(got_bits), bf16_to_f32(want_bits)
    extra = np.isnan(g) & ~np.isnan(w)
    assert not (extra & ~leak).any(), f"{(extra & ~leak).sum()} NaN outside the leak window"
    assert not (np.isnan(w) & ~np.isnan(g)).any(), "a NaN of the oracle is missing"
    keep = ~extra
    assert_precision(got_bits[keep], want_bits[keep], vmax[keep], precision)
    return int(extra.sum())


@pytest.mark.parametrize("precision", ["f16", "exact", "bf16"])
def test_nan_codes_propagate_like_the_oracle(precision):
    """NaN codes (e4m3 0x7F / 0xFF) in the pages.  A NaN K element makes every score of its
    key NaN: each row that sees the key is NaN in every channel, with lse2 -inf (the
    oracle's softmax denominator is NaN), and no other row changes (a masked score never
    reaches P).  A NaN V element makes its own channel NaN in the rows that see it; since
    the P.V product of a 64-key step multiplies the weight 0 of a key a row does not see
    by that key's V, rows before the key whose step holds it may also be NaN in that
    channel (as in tiled attention generally; the oracle skips such keys), and nothing
    else.  Checked for one step, and for ring attention over 3 shards in one launch and in
    separate launches merged through o_acc / lse2, where a NaN of the first step has to
    survive the later merges, which give it weight 0."""
    Hq, Hkv, P = 8, 2, 16
    n_q, q_pos0, lens = [48, 40], [0, 24], [48, 64]
    print(f"nan codes precision={precision}", flush=True)
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, n_q, q_pos0, lens, seed=31)
    pool[bt[0, 5 // P], 0, 0, 5 % P, 77] = 0x7F  # K of sequence 0, key 5, KV head 0, channel 77
    pool[bt[1, 30 // P], 1, 1, 30 % P, 17] = 0xFF  # V of sequence 1, key 30, KV head 1, channel 17
    kb, ke = np.zeros(2, np.int32), np.asarray(lens, np.int32)
    sm = float(np.float32(1.0 / np.sqrt(128)))
    want, wlse, err = O.paged_attention_prefill(bits16(q), cu, qp, pool, scales, bt, kb, ke, True, sm)
    assert err == 0
    w = bf16_to_f32(want)
    # the planted codes reach exactly the rows and channels described (causal: sequence 0's
    # rows from position 5 on, query heads 0-3; sequence 1's rows from position 30 on,
    # query heads 4-7, channel 17)
    assert np.isnan(w[5:48, 0:4]).all() and not np.isnan(w[0:5]).any()
    assert np.isnan(w[48 + 6:, 4:8, 17]).all() and not np.isnan(w[48:48 + 6]).any()
    assert np.isnan(w).sum() == 43 * 4 * 128 + 34 * 4
    assert np.isneginf(wlse[5:48, 0:4]).all()
    # where the NaN V may also show: sequence 1 (positions 24 + i), heads 4-7, channel 17,
    # rows less than 64 positions before key 30
    leak = np.zeros(w.shape, bool)
    leak[48:48 + 6, 4:8, 17] = True
    vm = vmax_rows(pool, scales, bt, cu, kb, ke, Hq)
    out, lse = run_step(q, pool, scales, bt, cu, qp, kb, ke, True, precision)
    torch.cuda.synchronize()
    n = assert_nan_leak_only_in_window(bits16(out), want, vm, precision, leak)
    g = lse.cpu().numpy()
    np.testing.assert_array_equal(np.isfinite(g), np.isfinite(wlse))
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    for single in (False, True):
        ring = kv.ring_attention_fp8(q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt), t(ke), ring_degree=3,
                                     causal=True, check=True, single_launch=single, precision=precision)
        torch.cuda.synchronize()
        n_ring = assert_nan_leak_only_in_window(bits16(ring), want, vm, precision, leak)
        print(f"  ring 3 single_launch={single}: {n_ring} NaN in the window (step: {n})", flush=True)


def test_prefill_flags_bad_pages():
    Hq, Hkv, P = 8, 2, 16
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, [40], [0], [64], seed=9, n_pages=8)
    bt = bt.copy()
    bt[0, 1] = 1000  # keys 16..31 on a page outside the pool
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    kb, ke = np.zeros(1, np.int32), np.full(1, 64, np.int32)
    with pytest.raises(ValueError, match="block table"):
        kv.paged_attention_prefill(q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt), t(kb), t(ke), causal=False,
                                   check=True)
    out = kv.paged_attention_prefill(q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt), t(kb), t(ke), causal=False)
    torch.cuda.synchronize()
    sm = float(np.float32(1.0 / np.sqrt(128)))
    want, _, err = O.paged_attention_prefill(bits16(q), cu, qp, pool, scales, bt, kb, ke, False, sm)
    assert err & 1
    assert_precision(bits16(out), want, vmax_rows(pool, scales, np.where(bt < 8, bt, 0), cu, kb, ke, Hq))


def test_prefill_kv_end_past_table_is_clipped_and_flagged():
    """kv_end beyond max_blocks * page_size: the kernel clips the key range to the table
    (as the oracle does), flags ZX_KERR_POS_RANGE, and check=True raises."""
    Hq, Hkv, P = 8, 2, 16
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, [40], [24], [64], seed=11)  # table holds 64 keys
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    kb, ke = np.zeros(1, np.int32), np.full(1, 80, np.int32)
    with pytest.raises(ValueError, match="max_blocks"):
        kv.paged_attention_prefill(q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt), t(kb), t(ke), causal=True,
                                   check=True)
    out = kv.paged_attention_prefill(q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt), t(kb), t(ke), causal=True)
    torch.cuda.synchronize()
    sm = float(np.float32(1.0 / np.sqrt(128)))
    want, _, err = O.paged_attention_prefill(bits16(q), cu, qp, pool, scales, bt, kb, ke, True, sm)
    assert err & 2
    assert_precision(bits16(out), want, vmax_rows(pool, scales, bt, cu, kb, np.full(1, 64, np.int32), Hq))


def test_prefill_rejects_bad_scales():
    Hq, Hkv, P = 8, 2, 16
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, [16], [0], [16], seed=12)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    kb, ke = np.zeros(1, np.int32), np.full(1, 16, np.int32)
    with pytest.raises(ValueError, match="scales_layer"):
        kv.paged_attention_prefill(q.to(DEV), t(cu), t(qp), t(pool), t(scales[:, :1]), t(bt), t(kb), t(ke))
    with pytest.raises(ValueError, match="scales_layer"):
        kv.paged_attention_prefill(q.to(DEV), t(cu), t(qp), t(pool), t(scales.astype(np.float64)), t(bt), t(kb),
                                   t(ke))


def test_prefill_flags_rows_beyond_max_q_per_seq():
    """A max_q_per_seq below a sequence's query count leaves the extra rows unwritten and is
    flagged (ZX_KERR_POS_RANGE); the covered rows are still right."""
    Hq, Hkv, P = 8, 2, 16
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, [200], [0], [200], seed=13)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    kb, ke = np.zeros(1, np.int32), np.full(1, 200, np.int32)
    with pytest.raises(ValueError, match="max_q_per_seq"):
        kv.paged_attention_prefill(q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt), t(kb), t(ke),
                                   max_q_per_seq=64, check=True)
    out = kv.paged_attention_prefill(q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt), t(kb), t(ke),
                                     max_q_per_seq=64)
    torch.cuda.synchronize()
    sm = float(np.float32(1.0 / np.sqrt(128)))
    want, _, err = O.paged_attention_prefill(bits16(q), cu, qp, pool, scales, bt, kb, ke, True, sm)
    assert err == 0
    covered = 64  # query tiles of 32 * 4 / G = 32 rows (G = 4 here): ceil(64 / 32) = 2 tiles cover rows 0..63
    assert_precision(bits16(out)[:covered], want[:covered], vmax_rows(pool, scales, bt, cu, kb, ke, Hq)[:covered])


def test_ring_degree_above_sequence_lengths():
    """Ring degree 8 over sequences of 3, 1 and 20 keys: most shards are empty (the first
    one too, which must still initialise the running output), the result is still full
    causal attention."""
    Hq, Hkv, P = 8, 2, 16
    lens = [3, 1, 20]
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, lens, [0, 0, 0], lens, seed=17)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    kl = np.asarray(lens, np.int32)
    sm = float(np.float32(1.0 / np.sqrt(128)))
    zeros = np.zeros(3, np.int32)
    want, _, err = O.paged_attention_prefill(bits16(q), cu, qp, pool, scales, bt, zeros, kl, True, sm)
    assert err == 0
    for single in (True, False):
        out = kv.ring_attention_fp8(q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt), t(kl), ring_degree=8,
                                    causal=True, check=True, single_launch=single)
        torch.cuda.synchronize()
        assert_precision(bits16(out), want, vmax_rows(pool, scales, bt, cu, zeros, kl, Hq))


def _f64_rows(q, pool, scales, bt, cu, qp, ranges, causal, sm):
    """Plain float64 attention over the given key ranges ([R][B] begin / end), and max |V|."""
    P, (n_rows, Hq, D), Hkv = pool.shape[3], q.shape, pool.shape[2]
    out = torch.zeros(q.shape, dtype=torch.float64, device=DEV)
    vmax = torch.zeros_like(out)
    for b in range(len(cu) - 1):
        t = torch.cat([torch.arange(lo[b], hi[b]) for lo, hi in ranges]).to(DEV)
        rows = slice(int(cu[b]), int(cu[b + 1]))
        pos = int(qp[b]) + torch.arange(rows.stop - rows.start, device=DEV)
        kv_ = pool[bt[b, t // P].long(), :, :, t % P].view(torch.float8_e4m3fn).float().double()
        kv_ = kv_ * scales.double()[None, :, :, None]  # [keys, 2, Hkv, D]
        for h in range(Hq):
            k, v = kv_[:, 0, h // (Hq // Hkv)], kv_[:, 1, h // (Hq // Hkv)]
            s = q[rows, h].double() @ k.t().contiguous() * sm
            if causal:
                s.masked_fill_(t[None, :] > pos[:, None], -np.inf)
            out[rows, h] = torch.nan_to_num(torch.softmax(s, dim=-1)) @ v
            vmax[rows, h] = v.abs().amax(dim=0)
    return out, vmax


@pytest.mark.parametrize("case", ["causal", "full", "ring", "gaps", "large_scores", "negative", "bad_page"])
@pytest.mark.parametrize("precision", ["f16", "bf16"])
def test_wide_prefill(case, precision):
    """The kernel with 64 rows per wave (four heads per KV head, at least a block per CU, room
    for 4,096 positions): ragged last tiles, steps cut by range ends, ranges that follow each
    other (walked as one) and ranges with gaps, running maxima that are outgrown again and
    again, negative scales of some heads' K and of others' V, and a bad page.  Bound: this
    module's, against float64."""
    Hq, Hkv, P = 32, 8, 48 if case == "gaps" else 16
    n_q, q_pos0, lens = [1030, 901, 1], [0, 700, 90], [1030, 1601, 91]
    print(f"wide prefill {case} {precision}", flush=True)
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, n_q, q_pos0, lens, seed=77)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    wide_bt = np.full((len(lens), 4096 // P + 1), -1, np.int32)
    wide_bt[:, :bt.shape[1]] = bt
    causal, sm = case != "full", float(np.float32(1.0 / np.sqrt(128)))
    if case == "large_scores":
        sm *= 12.0
    if case == "negative":
        scales *= np.array([[-1, 1, 1, -1, 1, 1, -1, 1], [1, -1, 1, -1, 1, 1, 1, -1]], np.float32)
    lens = np.asarray(lens)
    if case == "ring":
        ranges = [(lens * r // 5, lens * (r + 1) // 5) for r in range(5)]
    elif case == "gaps":
        ranges = [(lens * 0 + 5, lens // 3), (lens // 2, lens - 7)]
    else:
        ranges = [(lens * 0, lens)]
    q, pool, scales, bt = q.to(DEV), t(pool), t(scales), t(wide_bt)
    if case == "bad_page":
        bt[1, 20] = pool.shape[0]
        with pytest.raises(ValueError, match="block table"):
            kv.paged_attention_ring(q, t(cu), t(qp), pool, scales, bt, t(np.array([r[0] for r in ranges], np.int32)),
                                    t(np.array([r[1] for r in ranges], np.int32)), check=True, precision=precision)
        ranges = [(np.array([0, 0, 0]), np.array([lens[0], 20 * P, lens[2]])),
                  (np.array([0, 21 * P, 0]), np.array([0, lens[1], 0]))]
        kb, ke = t(np.zeros((1, 3), np.int32)), t(lens[None].astype(np.int32))
    else:
        kb, ke = (t(np.array([r[i] for r in ranges], np.int32)) for i in (0, 1))
    got, names = kernels_of(lambda: kv.paged_attention_ring(q, t(cu), t(qp), pool, scales, bt, kb, ke, causal=causal,
                                                            sm_scale=sm, check=case != "bad_page", precision=precision))
    assert "paged_prefill_wide_kernel" in names
    want, vmax = _f64_rows(q, pool, scales, bt, cu, qp, ranges, causal, sm)
    assert_precision(bits16(got), bits16(want.to(torch.bfloat16)), vmax.cpu().numpy(), precision)


@pytest.mark.parametrize("B,n,old,kernel", [
    (64, 32, 0, "mfma"), (32, 40, 4000, "mfma"), (64, 256, 0, "mfma"), (24, 600, 0, "mfma"),
    (4, 512, 0, "wide"), (10, 768, 0, "wide"), (32, 1024, 0, "wide"), (2, 1100, 900, "wide"),
])
def test_prefill_kernel_by_rows(B, n, old, kernel):
    """The 64-row kernel is for calls whose sequences have rows enough for its tiles, whatever
    the width of the table; others keep the 32-row kernel (64 sequences of 32 rows took 1.6
    times as long in half-empty tiles, short new sequences up to 1.3 times)."""
    Hq, Hkv, P = 32, 8, 16
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, [n] * B, [old] * B, [old + n] * B, seed=84)
    wide_bt = np.zeros((B, 8192 // P), np.int32)
    wide_bt[:, :bt.shape[1]] = bt
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    args = (q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(wide_bt), t(np.zeros(B, np.int32)),
            t(np.full(B, old + n, np.int32)))
    _, names = kernels_of(lambda: kv.paged_attention_prefill(*args, max_q_per_seq=n, check=True))
    assert f"paged_prefill_{kernel}_kernel" in names


def test_wide_prefill_flags_rows_beyond_max_q_per_seq():
    """As test_prefill_flags_rows_beyond_max_q_per_seq, for the 64-row kernel, whose last tile
    would hold 32 rows more: the rows up to a multiple of 32 are computed (as by the 32-row
    kernel), the others are left unwritten, and flagged."""
    Hq, Hkv, P, n = 32, 8, 16, 1088
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, [n, n], [0, 0], [n, n], seed=79)
    wide_bt = np.zeros((2, 4096 // P), np.int32)
    wide_bt[:, :bt.shape[1]] = bt
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    args = (q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(wide_bt), t(np.zeros(2, np.int32)), t(np.full(2, n, np.int32)))
    want, vmax = _f64_rows(args[0], args[3], args[4], args[5], cu, qp, [([0, 0], [n, n])], True,
                           float(np.float32(1.0 / np.sqrt(128))))
    out = torch.full(q.shape, 7.0, dtype=torch.bfloat16, device=DEV)
    _, names = kernels_of(lambda: kv.paged_attention_prefill(*args, out=out, max_q_per_seq=n - 32))
    assert "paged_prefill_wide_kernel" in names
    for at in (0, n):
        rows = slice(at, at + n - 32)
        assert_precision(bits16(out[rows]), bits16(want[rows].to(torch.bfloat16)), vmax[rows].cpu().numpy())
        assert (out[at + n - 32:at + n] == 7.0).all()
    for most, flagged in ((n - 32, True), (n - 31, False)):
        err = torch.zeros(1, dtype=torch.int32, device=DEV)
        kv.paged_attention_prefill(*args, max_q_per_seq=most, err=err)
        assert bool(err.item() & kv.N.ZX_KERR_POS_RANGE) == flagged


def test_wide_prefill_nan_v_reaches_no_further_than_the_32_row_kernels():
    """A NaN V code at key k makes its channel NaN in the rows from k on, and may do so in rows
    before it whose 32-row tile reaches the 64-key step that holds k.  Query positions start
    at 16, so that the first half of a 64-row tile ends before a step that its second half
    reaches."""
    Hq, Hkv, P, n, at = 32, 8, 16, 1088, 16
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, [n, n], [at, at], [at + n, at + n], seed=80)
    planted = {3: 100, 5: 127, 7: 500, 9: 1023, 11: 64}  # channel -> key, of sequence 0's KV head 2
    for ch, k in planted.items():
        pool[bt[0, k // P], 1, 2, k % P, ch] = 0x7F
    wide_bt = np.zeros((2, 4096 // P), np.int32)
    wide_bt[:, :bt.shape[1]] = bt
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    got, names = kernels_of(lambda: kv.paged_attention_prefill(
        q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(wide_bt), t(np.zeros(2, np.int32)),
        t(np.full(2, at + n, np.int32)), max_q_per_seq=n))
    assert "paged_prefill_wide_kernel" in names
    nan = torch.isnan(got.float()).cpu().numpy()
    row = np.arange(n)
    may = np.zeros_like(nan)
    for ch, k in planted.items():
        assert nan[:n][row + at >= k][:, 8:12, ch].all()
        reaches = at + np.minimum(row // 32 * 32 + 31, n - 1) >= k // 64 * 64
        may[:n, 8:12, ch] = reaches[:, None]
    assert not (nan & ~may).any(), np.argwhere(nan & ~may)[:5]


@pytest.mark.parametrize("kind", ["negative_scale"])
def test_wide_prefill_takes_the_overlapped_steps(kind):
    """Calls that once sent every step through the kernel's masked path (1.9 times the time)
    take no longer than the plain call."""
    Hq, Hkv, P, n = 32, 8, 16, 4096
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, [n, n], [0, 0], [n, n], seed=81)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    args = [q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt), t(np.zeros((1, 2), np.int32)),
            t(np.full((1, 2), n, np.int32))]
    sm = 1e-4  # scores of a few log2 units: no step is repeated

    def call(sign=1.0):
        return kv.paged_attention_ring(*args, causal=False, sm_scale=sign * sm, max_q_per_seq=n)

    assert "paged_prefill_wide_kernel" in kernels_of(call)[1]
    plain = min(least_us(call), least_us(call))
    odd = min(least_us(lambda: call(-1.0)), least_us(lambda: call(-1.0)))
    print(f"plain {plain:.0f} us, {kind} {odd:.0f} us", flush=True)
    assert odd <= 1.3 * plain


def test_wide_prefill_keys_above_the_first_ones():
    """All keys but the first 64 score 6 log2 units above those: within the slack of a running
    maximum, but the sums of their weights are not.  The maxima follow, so the call takes no
    longer than with the keys 1 above (every step was made twice where they did not: 1.6
    times), and the rows are the weighted means."""
    Hq, Hkv, P, n = 32, 8, 16, 4096
    g = torch.Generator(device=DEV).manual_seed(4)
    pool = torch.zeros((2 * n // P, 2, Hkv, P, 128), dtype=torch.uint8, device=DEV)
    pool[:, 1] = torch.where(torch.rand(pool[:, 1].shape, generator=g, device=DEV) < 0.5, 0x38, 0x30).to(torch.uint8)
    pool[:, 0, :, :, 0] = 0x38
    bt = torch.arange(2 * n // P, dtype=torch.int32, device=DEV).view(2, -1)
    pool[bt[:, :4].flatten().long(), 0] = 0
    q = torch.zeros((2 * n, Hq, 128), dtype=torch.bfloat16, device=DEV)
    q[..., 0] = 1.0
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    args = (q, i32([0, n, 2 * n]), i32([0, 0]), pool, torch.ones((2, Hkv), device=DEV), bt, i32([[0, 0]]), i32([[n, n]]))
    v = pool[bt.long(), 1].view(torch.float8_e4m3fn).float().double()  # [2, pages, Hkv, P, 128]
    v = v.permute(0, 2, 1, 3, 4).reshape(2, Hkv, n, 128)
    took = {}
    for above in (1, 6, 1, 6):
        call = lambda: kv.paged_attention_ring(*args, causal=False, sm_scale=above * float(np.log(2.0)), max_q_per_seq=n)  # noqa: E731,B023
        got, names = kernels_of(call)
        assert "paged_prefill_wide_kernel" in names
        w = torch.ones(n, dtype=torch.float64, device=DEV)
        w[:64] = 2.0 ** -above
        want = ((w[None, None, :, None] * v).sum(2) / w.sum()).repeat_interleave(Hq // Hkv, 1)  # [2, Hq, 128]
        assert (got.view(2, n, Hq, 128).double() - want[:, None]).abs().max() <= 2.0 ** -8
        took[above] = min(took.get(above, 1e9), least_us(call))
    print(f"1 above: {took[1]:.0f} us, 6 above: {took[6]:.0f} us", flush=True)
    assert took[6] <= 1.3 * took[1], took


@pytest.mark.parametrize("below", [6, 14, 20, 22, 24])
def test_wide_prefill_weights_far_below_the_largest(below):
    """One key whose score lies ``below`` log2 units above all 65,535 others: their weights,
    subnormal in fp16 from 22 on (2^(7 - 22) < 2^-14), count in the row sums as they do in
    P.V.  They are powers of two, so P is exact and the result is the exact value within an
    ulp of bf16 (at 22 they are 1.6% of a row's sum, four ulps)."""
    Hq, Hkv, P, n_keys, n_q = 32, 8, 16, 65536, 2112
    g = torch.Generator(device=DEV).manual_seed(1)
    pool = torch.zeros((n_keys // P, 2, Hkv, P, 128), dtype=torch.uint8, device=DEV)
    pool[:, 1] = torch.where(torch.rand(pool[:, 1].shape, generator=g, device=DEV) < 0.5, 0x38, 0x30).to(torch.uint8)
    pool[0, 0, :, 0, 0] = 0x38  # key 0: 1.0 in channel 0, as every query
    q = torch.zeros((n_q, Hq, 128), dtype=torch.bfloat16, device=DEV)
    q[..., 0] = 1.0
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    got, names = kernels_of(lambda: kv.ring_attention_fp8(
        q, i32([0, n_q]), i32([n_keys - n_q]), pool, torch.ones((2, Hkv), device=DEV),
        torch.arange(n_keys // P, dtype=torch.int32, device=DEV)[None], i32([n_keys]), 1, causal=False,
        sm_scale=below * float(np.log(2.0)), max_q_per_seq=n_q))
    assert "paged_prefill_wide_kernel" in names
    v = pool[:, 1].view(torch.float8_e4m3fn).float().double().permute(1, 0, 2, 3).reshape(Hkv, n_keys, 128)
    w = torch.full((n_keys,), 2.0 ** -below, dtype=torch.float64, device=DEV)
    w[0] = 1.0
    want = (w[None, :, None] * v).sum(1) / w.sum()  # between 0.5 and 1: an ulp is 2^-8
    diff = (got.double() - want.repeat_interleave(Hq // Hkv, 0)[None]).abs().max().item()
    assert diff <= 2.0 ** -8, diff


@pytest.mark.parametrize("Hq,Hkv,P,n_q,q_pos0,causal,precision", [
    (32, 8, 16, [5, 1, 40], [1500, 600, 2100], True, "f16"),   # several parts; sequences of different lengths
    (8, 2, 16, [33], [1023], True, "exact"),                   # a part per 8 steps, tiles of 32 rows and 1
    (4, 4, 48, [130, 3], [2000, 12], True, "bf16"),            # one head per KV head; a sequence with keys for one part
    (6, 3, 32, [17, 64], [0, 1500], False, "f16"),             # two heads per KV head; every row sees every key
])
def test_prefill_in_parts(Hq, Hkv, P, n_q, q_pos0, causal, precision):
    """Calls with few query tiles: several blocks share a tile's keys and their parts are
    combined; with a ring's contiguous shards and with a gap between two ranges.  Rows beyond
    max_q_per_seq stay unwritten.  Bound: this module's, against float64 (the combination is
    an average under the same weights in fp32, far below it)."""
    lens = np.asarray([p + n for p, n in zip(q_pos0, n_q)])
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, n_q, q_pos0, lens.tolist(), seed=5 * Hq + P)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    q, pool, scales, bt = q.to(DEV), t(pool), t(scales), t(bt)
    sm = float(np.float32(1.0 / np.sqrt(128)))
    for ranges in ([(lens * r // 3, lens * (r + 1) // 3) for r in range(3)], [(lens * 0 + 3, lens // 3), (lens // 2, lens)]):
        kb, ke = (t(np.array([r[i] for r in ranges], np.int32)) for i in (0, 1))
        got, names = kernels_of(lambda: kv.paged_attention_ring(q, t(cu), t(qp), pool, scales, bt, kb, ke, causal=causal,  # noqa: B023
                                                                sm_scale=sm, check=True, precision=precision))
        assert "prefill_combine_kernel" in names
        want, vmax = _f64_rows(q, pool, scales, bt, cu, qp, ranges, causal, sm)
        assert_precision(bits16(got), bits16(want.to(torch.bfloat16)), vmax.cpu().numpy(), precision)
    zero, end = t(np.zeros(len(n_q), np.int32)), t(lens.astype(np.int32))
    out = torch.full(q.shape, 7.0, dtype=torch.bfloat16, device=DEV)
    kv.paged_attention_prefill(q, t(cu), t(qp), pool, scales, bt, zero, end, causal=causal, out=out, max_q_per_seq=1,
                               precision=precision)
    rows = 32 * 4 // (4 if Hq // Hkv % 4 == 0 else 2 if Hq // Hkv % 2 == 0 else 1)  # of the one tile that is computed
    for b, n in enumerate(n_q):
        assert (out[int(cu[b]) + rows:int(cu[b]) + n] == 7.0).all()


@pytest.mark.parametrize("Hq,n_q,q_pos0,causal", [
    (32, [64], [448], True),              # one part a tile: written by its own block
    (32, [64, 64, 64, 64], [0] * 4, True),
    (32, [70, 1, 33], [0, 3000, 900], True),  # one part, several, and in between
    (16, [130, 40], [0, 2000], False),
])
def test_parts_follow_the_lengths(Hq, n_q, q_pos0, causal):
    """A block table far wider than the sequences gives room for parts that the real lengths do
    not need: the rows are right (in NaN-filled outputs), and the call takes about as long as
    with the exact table (parts of the table's width: 5 times as long)."""
    Hkv, P = 8, 16
    lens = [p + n for p, n in zip(q_pos0, n_q)]
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, n_q, q_pos0, lens, seed=83)
    wide_bt = np.full((len(lens), 32768 // P), -1, np.int32)
    wide_bt[:, :bt.shape[1]] = bt
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    q, pool, scales = q.to(DEV), t(pool), t(scales)
    zero, end = t(np.zeros(len(n_q), np.int32)), t(np.asarray(lens, np.int32))
    want, vmax = _f64_rows(q, pool, scales, t(bt), cu, qp, [([0] * len(n_q), lens)], causal, 128 ** -0.5)
    took = {}
    for name, table in (("exact", t(bt)), ("wide", t(wide_bt))) * 2:
        out = torch.full(q.shape, float("nan"), dtype=torch.bfloat16, device=DEV)
        call = lambda: kv.paged_attention_prefill(q, t(cu), t(qp), pool, scales, table, zero, end, causal=causal,  # noqa: E731,B023
                                                  out=out, max_q_per_seq=max(n_q))  # noqa: B023
        names = kernels_of(call)[1]
        assert "prefill_combine_kernel" in names or name == "exact"
        assert_precision(bits16(out), bits16(want.to(torch.bfloat16)), vmax.cpu().numpy())
        graph = torch.cuda.CUDAGraph()  # the launches without the host's part
        args = (q, t(cu), t(qp), pool, scales, table, zero, end)
        with torch.cuda.graph(graph):
            for _ in range(10):
                kv.paged_attention_prefill(*args, causal=causal, out=out, max_q_per_seq=max(n_q))
        out.fill_(float("nan"))
        took[name] = min(took.get(name, 1e9), least_us(graph.replay) / 10)
        assert_precision(bits16(out), bits16(want.to(torch.bfloat16)), vmax.cpu().numpy())
    print(f"exact table {took['exact']:.1f} us, 32k table {took['wide']:.1f} us", flush=True)
    assert took["wide"] <= 1.1 * took["exact"] + 8


@pytest.mark.parametrize("ring", [8, 64])
def test_parts_of_a_ring_are_equal(ring):
    """The parts of a tile's keys are equal runs of all its steps, also where a ring's shards
    have fewer steps than there are parts: such a ring takes about as long as one range (dealt
    shard by shard, one part of a ring of 64 got every step: 3 times the time)."""
    Hq, Hkv, P, n, old = 32, 8, 16, 64, 4032
    q, pool, scales, bt, cu, qp = make(Hq, Hkv, P, [n], [old], [old + n], seed=82)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    args = [q.to(DEV), t(cu), t(qp), t(pool), t(scales), t(bt)]
    want, vmax = _f64_rows(args[0], args[3], args[4], args[5], cu, qp, [([0], [old + n])], True, 128 ** -0.5)
    took = {}
    for R in (1, ring, 1, ring):
        kb, ke = (torch.arange(R, dtype=torch.int32, device=DEV)[:, None] + i for i in (0, 1))
        kb, ke = kb * ((old + n) // R), ke * ((old + n) // R)
        call = lambda: kv.paged_attention_ring(*args, kb, ke, max_q_per_seq=n)  # noqa: E731,B023
        got, names = kernels_of(call)
        assert "prefill_combine_kernel" in names
        assert_precision(bits16(got), bits16(want.to(torch.bfloat16)), vmax.cpu().numpy())
        took[R] = min(took.get(R, 1e9), least_us(call))
    print(f"one range {took[1]:.0f} us, ring of {ring} {took[ring]:.0f} us", flush=True)
    assert took[ring] <= 1.6 * took[1]


def test_ring_shard_bounds_match_torch():
    """The shard bounds' kernel against the integer expression, negative and large lengths
    among them; a kv_len of another dtype gives the same attention."""
    lens = torch.tensor([0, 1, 7, 8191, 2**31 - 1, -5], dtype=torch.int32, device=DEV)
    for R in (1, 3, 70):
        row = 8
        begin = torch.full((R, row), -99, dtype=torch.int32, device=DEV)
        end = begin.clone()
        lib = kv.N.load()
        kv.N.check(lib.zx_ring_shard_bounds(kv.N.ptr(lens), 6, R, row, kv.N.ptr(begin), kv.N.ptr(end),
                                            kv.N.stream_ptr(DEV)), "bounds")
        want = lens.to(torch.int64)[None] * torch.arange(R + 1, device=DEV)[:, None] // R
        assert torch.equal(begin[:, :6].long(), want[:-1]) and torch.equal(end[:, :6].long(), want[1:])
        assert (begin[:, 6:] == -99).all()
    c = _ring_case()
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    args = (c["q"].to(DEV), t(c["cu"]), t(c["qp"]), t(c["pool"]), t(c["scales"]), t(c["bt"]))
    a = kv.ring_attention_fp8(*args, t(c["lens"]), 3)
    b = kv.ring_attention_fp8(*args, t(c["lens"]).long(), 3)
    assert torch.equal(a, b)
