"""GPU decode attention from FP8 pages (zx_paged_attention_decode) against the C oracle.

The oracle evaluates softmax(sm_scale q K^T) V in double on the decoded codes times the
per-head scales and rounds once to bf16 (it is pinned bit-exact against torch float64 in
tests/test_oracle.py).  The kernel computes in fp32 with a split online softmax and
exp2, so the tolerance is one bf16 ulp of the exact value plus the fp32 accumulation
error of a weighted mean of the V column (which matters only where the output cancels
to far below the V values):
    |got - want| <= ulp(|want|) + 2^-17 * max_t |V_t[d]|,   ulp(x) = 2^(floor(log2 x) - 7)
(values below 2^-100 take ulp 2^-107; 2^-17 bounds the fp32 error of summing up to 4096
weighted terms in the kernel's order), NaN compared as a class.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from zenyx_amd import kv

pytestmark = pytest.mark.gpu


def bits16(t: torch.Tensor) -> np.ndarray:
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def bf16_to_f32(b: np.ndarray) -> np.ndarray:
    return (b.astype(np.uint32) << 16).view(np.float32)


def kernels_of(fn):
    """fn's result and the names of the kernels it launched, so that a test of one kernel
    fails when the library's rule sends its call to another."""
    for _ in range(3):  # (a first trace of a process may come back empty)
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
            out = fn()
            torch.cuda.synchronize()
        names = " ".join(e.key for e in prof.key_averages())
        if "kernel" in names:
            break
    return out, names


def least_us(call):
    took = []
    for _ in range(8):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        call()
        b.record()
        b.synchronize()
        took.append(a.elapsed_time(b) * 1e3)
    return min(took)


def v_colmax(pool, scales, bt, lens, Hq):
    """max_t |V_t[d]| over each sequence's positions with a valid page: [B, Hq, D]."""
    n_pages, _, Hkv, P, D = pool.shape
    dec = np.abs(O.e4m3_decode(np.arange(256, dtype=np.uint8)).astype(np.float64))
    out = np.zeros((len(lens), Hq, D))
    for b, n in enumerate(lens):
        t = np.arange(n)
        pages = bt[b, t // P]
        ok = (pages >= 0) & (pages < n_pages)
        t, pages = t[ok], pages[ok]
        for hq in range(Hq):
            h = hq // (Hq // Hkv)
            if len(t):
                out[b, hq] = np.nanmax(dec[pool[pages, 1, h, t % P, :]], axis=0) * abs(float(scales[1, h]))
    return out


def assert_within_bound(got_bits: np.ndarray, want_bits: np.ndarray, vmax: np.ndarray, e: float, ulps: int = 1):
    """|got - want| <= ``ulps`` bf16 ulps of want + e * max|V| elementwise (NaN as a class)."""
    g, w = bf16_to_f32(got_bits), bf16_to_f32(want_bits)
    g_nan, w_nan = np.isnan(g), np.isnan(w)
    np.testing.assert_array_equal(g_nan, w_nan)
    g, w, vm = g[~g_nan].astype(np.float64), w[~w_nan].astype(np.float64), vmax[~w_nan]
    mag = np.maximum(np.abs(w), 2.0 ** -100)
    tol = ulps * np.exp2(np.floor(np.log2(mag)) - 7) + e * vm
    bad = np.abs(g - w) > tol
    assert not bad.any(), f"{bad.sum()} of {bad.size} beyond tolerance, e.g. got {g[bad][:4]} want {w[bad][:4]}"
    return float(np.max(np.abs(g - w) / np.maximum(vm, 1e-30))) if g.size else 0.0


def assert_within_one_ulp(got_bits: np.ndarray, want_bits: np.ndarray, vmax: np.ndarray):
    """The exact kernels' bound: one bf16 ulp + 2^-17 max|V|."""
    return assert_within_bound(got_bits, want_bits, vmax, 2.0 ** -17)


def make_case(Hq, Hkv, D, P, lens, seed, n_pages=None, nan_codes=False):
    rng = np.random.default_rng(seed)
    lens = np.asarray(lens, np.int32)
    B = len(lens)
    max_blocks = max(1, (int(lens.max()) + P - 1) // P)
    n_pages = n_pages or B * max_blocks + 5
    pool = rng.integers(0, 256, (n_pages, 2, Hkv, P, D), dtype=np.uint8)
    if not nan_codes:
        pool[(pool & 0x7F) == 0x7F] = 0x3A
    perm = rng.permutation(n_pages)
    bt = perm[:B * max_blocks].reshape(B, max_blocks).astype(np.int32)
    scales = rng.uniform(1e-3, 0.05, (2, Hkv)).astype(np.float32)
    q = torch.from_numpy(rng.standard_normal((B, Hq, D)).astype(np.float32)).to(torch.bfloat16)
    return q, pool, scales, bt, lens


@pytest.mark.parametrize("Hq,Hkv,D,P,lens", [
    (32, 8, 128, 16, [0, 1, 15, 16, 17, 1023, 1024, 1025, 3000]),  # 4 query heads per block
    (8, 8, 64, 16, [5, 64, 2100]),                                  # no grouping, D = 64
    (12, 4, 256, 32, [700, 31, 2049]),                              # groups of 3 (one head per block)
    (16, 8, 128, 5, [1, 333, 1500]),                                # page size 5, pairs of heads
    (8, 8, 128, 32, [40, 1, 2222]),                                 # matrix-core variant, one head
    (16, 8, 128, 16, [17, 4000]),                                   # matrix-core variant, pairs
])
def test_paged_attention_decode_matches_oracle(dev, Hq, Hkv, D, P, lens):
    q, pool, scales, bt, lens = make_case(Hq, Hkv, D, P, lens, seed=Hq + D + P)
    sm = 1.0 / np.sqrt(D)
    want, werr = O.paged_attention_decode(bits16(q), pool, scales, bt, lens, sm)
    assert werr == 0
    got = kv.paged_attention_decode(q.to(dev), torch.from_numpy(pool).to(dev), torch.from_numpy(scales).to(dev),
                                    torch.from_numpy(bt).to(dev), torch.from_numpy(lens).to(dev), check=True)
    assert_within_one_ulp(bits16(got), want, v_colmax(pool, scales, bt, lens, Hq))
    assert not bits16(got)[lens == 0].any()  # empty sequences give zeros


def test_paged_attention_decode_large_scores_and_custom_scale(dev):
    """Large logits (scale 8x sm_scale) stress the running-max rescaling across splits."""
    q, pool, scales, bt, lens = make_case(32, 8, 128, 16, [4096, 2000, 9], seed=5)
    scales[0] *= 20.0
    sm = 8.0 / np.sqrt(128)
    want, _ = O.paged_attention_decode(bits16(q), pool, scales, bt, lens, sm)
    got = kv.paged_attention_decode(q.to(dev), torch.from_numpy(pool).to(dev), torch.from_numpy(scales).to(dev),
                                    torch.from_numpy(bt).to(dev), torch.from_numpy(lens).to(dev), sm_scale=sm)
    assert_within_one_ulp(bits16(got), want, v_colmax(pool, scales, bt, lens, 32))


@pytest.mark.parametrize("Hq,Hkv,D", [(32, 8, 128), (8, 8, 64)])
def test_paged_attention_decode_negative_scales(dev, Hq, Hkv, D):
    """Scales of either sign (a static scale may be negative): K heads 0, 2, .. and V heads
    1, 3, .. negated, so scores and values change sign per head (matrix-core kernel for
    D = 128, VALU kernel for D = 64)."""
    q, pool, scales, bt, lens = make_case(Hq, Hkv, D, 16, [1, 300, 2500], seed=13)
    scales[0, 0::2] *= -1.0
    scales[1, 1::2] *= -1.0
    sm = 1.0 / np.sqrt(D)
    want, werr = O.paged_attention_decode(bits16(q), pool, scales, bt, lens, sm)
    assert werr == 0
    got = kv.paged_attention_decode(q.to(dev), torch.from_numpy(pool).to(dev), torch.from_numpy(scales).to(dev),
                                    torch.from_numpy(bt).to(dev), torch.from_numpy(lens).to(dev), check=True)
    assert_within_one_ulp(bits16(got), want, v_colmax(pool, scales, bt, lens, Hq))


@pytest.mark.parametrize("D", [64, 128])
def test_paged_attention_decode_nan_codes_and_bad_pages(dev, D):
    """NaN codes make the affected heads NaN; an out-of-range page id is skipped and flagged
    (D = 64: VALU kernel, D = 128: matrix-core kernel)."""
    q, pool, scales, bt, lens = make_case(8, 2, D, 16, [100, 200, 50], seed=6)
    pool[bt[1, 3], 0, 1, 4, 7] = 0x7F  # a NaN code in sequence 1, kv head 1
    bt_bad = bt.copy()
    bt_bad[2, 1] = pool.shape[0] + 10
    want, werr = O.paged_attention_decode(bits16(q), pool, scales, bt_bad, lens, 0.125)
    assert werr == 1
    args = (q.to(dev), torch.from_numpy(pool).to(dev), torch.from_numpy(scales).to(dev),
            torch.from_numpy(bt_bad).to(dev), torch.from_numpy(lens).to(dev))
    with pytest.raises(ValueError, match="block table"):
        kv.paged_attention_decode(*args, sm_scale=0.125, check=True)
    got = kv.paged_attention_decode(*args, sm_scale=0.125)
    assert_within_one_ulp(bits16(got), want, v_colmax(pool, scales, bt_bad, lens, 8))
    assert np.isnan(bf16_to_f32(bits16(got)[1, 4:8])).all()


@pytest.mark.parametrize("Hq,Hkv,D,P,lens", [
    (64, 8, 128, 16, [127, 128, 129, 0, 700]),     # 8 heads per block; sequence ends on and beside a unit's end
    (32, 1, 64, 32, [513, 1, 0, 0, 255, 256]),     # 32 heads: two blocks of 16; empty sequences inside a run
    (20, 4, 128, 48, [31, 33, 2000]),              # 5 heads per block
    (16, 4, 64, 16, [int(v) for v in np.random.default_rng(3).integers(0, 300, 67)]),   # > 64 sequences
    (4, 4, 128, 16, [int(v) for v in np.random.default_rng(4).integers(0, 900, 300)]),  # > 256, one head per block
    (8, 2, 128, 16, [int(v) for v in np.random.default_rng(5).integers(0, 500, 140)]),  # whole sequences per block
    (8, 2, 256, 16, [0, 64, 65, 1000]),
])
def test_paged_attention_decode_runs_and_segments(dev, Hq, Hkv, D, P, lens):
    """The positions of all sequences are dealt to the blocks in equal runs of units (128
    positions; 64 - 256 without matrix cores): runs that hold several sequences, sequences
    over several runs, unit and tile edges, empty sequences, and more sequences than one wave
    (64) or one block (256) looks through at a time.  Bound: this module's (fp32 sums)."""
    q, pool, scales, bt, lens = make_case(Hq, Hkv, D, P, lens, seed=Hq + D + len(lens))
    sm = 1.0 / np.sqrt(D)
    want, werr = O.paged_attention_decode(bits16(q), pool, scales, bt, lens, sm)
    assert werr == 0
    got = kv.paged_attention_decode(q.to(dev), torch.from_numpy(pool).to(dev), torch.from_numpy(scales).to(dev),
                                    torch.from_numpy(bt).to(dev), torch.from_numpy(lens).to(dev), check=True)
    assert_within_one_ulp(bits16(got), want, v_colmax(pool, scales, bt, lens, Hq))
    assert not bits16(got)[lens == 0].any()


@pytest.mark.parametrize("Hq,Hkv", [(8, 8), (16, 8), (32, 8), (128, 8)])
def test_decode_head_dim_64_weights_keep_32_bits(dev, Hq, Hkv):
    """Pairs of keys whose weights differ by 2^-13 with values +448 and -448: the values cancel,
    and what is left shows the error of the weights.  With 32-bit weights and products it
    is at most that of exp2 (an ulp), of its argument (below 4, rounded to 2^-23) and of
    the sums, 2^-20.5 max|V| together; weights in two bf16 terms give 2^-18.7."""
    B, n, D, P = 64, 8, 64, 16
    g = torch.Generator().manual_seed(Hq)
    k = torch.zeros((B, Hkv, P, D))
    k[..., 0] = torch.randint(-8, 9, (B, Hkv, P // 2), generator=g).repeat_interleave(2, 2) / 8.0  # e4m3 values
    k[..., 1::2, 1] = 1.0
    v = torch.randint(0, 2, (B, Hkv, P // 2, D), generator=g).repeat_interleave(2, 2) * 2.0 - 1.0
    v[..., 1::2, :] *= -1.0
    pool = torch.stack([k, 448.0 * v], 1).to(torch.float8_e4m3fn).view(torch.uint8)  # a page per sequence
    q = torch.zeros((B, Hq, D))
    q[..., 0] = torch.rand((B, Hq), generator=g) * 4.0 - 2.0
    q[..., 1] = 2.0 ** -13
    q = q.to(torch.bfloat16)
    got = kv.paged_attention_decode(q.to(dev), pool.to(dev), torch.ones((2, Hkv), device=dev),
                                    torch.arange(B, dtype=torch.int32, device=dev)[:, None].contiguous(),
                                    torch.full((B,), n, dtype=torch.int32, device=dev), sm_scale=1.0)
    rep = Hq // Hkv
    kd, vd = (t[:, :, :n].double().repeat_interleave(rep, 1) for t in (k, 448.0 * v))
    w = torch.softmax((q.double()[:, :, None] * kd).sum(-1), -1)
    want = (w[..., None] * vd).sum(2)
    off = (got.cpu().double() - want).abs() - want.abs() * 2.0 ** -8  # the rounding to bf16: half an ulp
    worst = off.max().item() / 448.0
    print(f"Hq {Hq}: 2^{np.log2(max(worst, 1e-12)):.1f} max|V|", flush=True)
    assert worst <= 2.0 ** -20.5


@pytest.mark.parametrize("Hq,Hkv,D,kernel", [
    (38, 2, 64, "partial"), (38, 2, 128, "partial"),  # 19 query heads per kv head: one per block
    (8, 8, 64, "partial"), (36, 2, 64, "mfma"), (68, 2, 64, "mfma"), (26, 2, 128, "mfma"),  # 9, 2 and 13 per block
])
def test_decode_kernel_by_heads(dev, Hq, Hkv, D, kernel):
    """The matrix-core kernel is for blocks of several query heads; one head per block goes to
    the other.  Both against the oracle."""
    q, pool, scales, bt, lens = make_case(Hq, Hkv, D, 16, [700, 17, 1], seed=Hq + D)
    want, _ = O.paged_attention_decode(bits16(q), pool, scales, bt, lens, 1.0 / np.sqrt(D))
    args = [t.to(dev) for t in (q, *map(torch.from_numpy, (pool, scales, bt, lens)))]
    got, names = kernels_of(lambda: kv.paged_attention_decode(*args, check=True))
    assert_within_one_ulp(bits16(got), want, v_colmax(pool, scales, bt, lens, Hq))
    assert f"paged_decode_{kernel}_kernel" in names


@pytest.mark.parametrize("D,P", [(64, 24), (128, 4), (256, 2)])
def test_decode_four_heads_share_their_pages(dev, D, P):
    """Pages that are no multiple of a wave's pass: a block of four query heads reads its pages
    once, as one of two does, and takes at most 1.5 times as long (1.9 times where its
    registers left one wave per SIMD)."""
    rng = np.random.default_rng(7)
    lens = rng.integers(2048, 8192, 64)
    took = {}
    for Hq in (16, 32):
        need = -(-lens // P)
        bt = np.zeros((64, need.max()), np.int32)
        for b, first in enumerate(np.cumsum(need) - need):
            bt[b, :need[b]] = first + np.arange(need[b])
        Hkv = 8 if D < 256 else 4
        pool = torch.randint(0, 0x70, (int(need.sum()), 2, Hkv, P, D), dtype=torch.uint8, device=dev)
        args = [torch.randn((64, Hq * Hkv // 8, D), device=dev).to(torch.bfloat16), pool, torch.full((2, Hkv), 0.01, device=dev),
                torch.from_numpy(bt).to(dev), torch.from_numpy(lens.astype(np.int32)).to(dev)]
        took[Hq] = least_us(lambda: kv.paged_attention_decode(*args))  # noqa: B023
    print(f"two heads {took[16]:.0f} us, four {took[32]:.0f} us", flush=True)
    assert took[32] <= 1.5 * took[16]


@pytest.mark.parametrize("Hq,Hkv,D,P", [(32, 8, 128, 16), (12, 12, 64, 16), (16, 4, 256, 8), (8, 2, 64, 24)])
@pytest.mark.parametrize("lens", ["few_short", "few", "whole_64", "runs_64", "whole_65", "runs_65", "many_short",
                                  "many", "one_long"])
def test_decode_dealt_by_the_lengths(dev, Hq, Hkv, D, P, lens):
    """The positions are dealt to the blocks in equal runs or as whole sequences, by the lengths
    that the device reads (up to 64 sequences in every wave, more by a kernel of its own):
    every way of it against the oracle, with empty sequences among them, and in a graph
    that is replayed with other lengths."""
    rng = np.random.default_rng(len(lens) + D)
    n = {"few_short": rng.integers(0, 200, 5), "few": rng.integers(0, 3000, 9), "whole_64": rng.integers(0, 130, 64),
         "runs_64": rng.integers(0, 700, 64), "whole_65": rng.integers(0, 130, 65), "runs_65": rng.integers(0, 700, 65),
         "many_short": rng.integers(0, 40, 1500), "many": rng.integers(0, 300, 300),
         "one_long": np.r_[rng.integers(0, 20, 40), 6000, rng.integers(0, 20, 90)]}[lens].astype(np.int32)
    if lens.startswith("runs"):
        n[7] = 5000  # the longest is far above an equal share
    B, width = len(n), -(-6200 // P) if B_wide(lens) else -(-int(n.max() + 1) // P)
    need = np.maximum(-(-n // P), 1)
    pages = int(need.sum()) + 3
    pool = rng.integers(0, 256, (pages, 2, Hkv, P, D), dtype=np.uint8)
    pool[(pool & 0x7F) == 0x7F] = 0x3A
    bt = np.full((B, width), -1, np.int32)
    perm = rng.permutation(pages).astype(np.int32)
    for b, first in enumerate(np.cumsum(need) - need):
        bt[b, :need[b]] = perm[first:first + need[b]]
    scales = rng.uniform(1e-3, 0.05, (2, Hkv)).astype(np.float32)
    q = torch.from_numpy(rng.standard_normal((B, Hq, D)).astype(np.float32)).to(torch.bfloat16)
    qd, pd, sd, bd, nd = (t.to(dev) for t in (q, *map(torch.from_numpy, (pool, scales, bt, n))))
    other = np.minimum(n, rng.permutation(n)).astype(np.int32)  # within every sequence's pages
    want = {}
    for key, v in (("n", n), ("other", other)):
        want[key], err = O.paged_attention_decode(bits16(q), pool, scales, bt, v, 1.0 / np.sqrt(D))
        assert err == 0
        got = kv.paged_attention_decode(qd, pd, sd, bd, torch.from_numpy(v).to(dev), check=True)
        assert_within_one_ulp(bits16(got), want[key], v_colmax(pool, scales, bt, v, Hq))
        assert not bits16(got)[v == 0].any()
    out = torch.empty_like(qd)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        kv.paged_attention_decode(qd, pd, sd, bd, nd, out=out)
    for key, v in (("other", other), ("n", n), ("other", other)):
        nd.copy_(torch.from_numpy(v))
        out.fill_(float("nan"))
        graph.replay()
        assert_within_one_ulp(bits16(out), want[key], v_colmax(pool, scales, bt, v, Hq))


def B_wide(lens):
    """Lengths that the host, which knows the table's width only, cannot deal as whole sequences."""
    return lens not in ("few", "many")


def test_decode_work_grows_with_the_sequences(dev):
    """4,096 sequences take about 16 times as long as 256 (57 times where every block went
    over all lengths)."""
    took = {}
    for B in (256, 4096):
        pages = B * 38
        pool = torch.randint(0, 0x70, (pages, 2, 8, 16, 128), dtype=torch.uint8, device=dev)
        args = [torch.randn((B, 32, 128), device=dev).to(torch.bfloat16), pool, torch.full((2, 8), 0.01, device=dev),
                torch.arange(pages, dtype=torch.int32, device=dev).view(B, 38).repeat(1, 2),
                torch.full((B,), 600, dtype=torch.int32, device=dev)]
        took[B] = least_us(lambda: kv.paged_attention_decode(*args))  # noqa: B023
    print(f"256: {took[256]:.0f} us, 4,096: {took[4096]:.0f} us", flush=True)
    assert took[4096] <= 24 * took[256]
