"""The matrix-core kernels of the shape-general attention at the sizes where
their tiles, windows and context parts end, over every form that selects a
path, and rows whose values are not finite."""
import numpy as np
import pytest
import torch

import oracle as O
import rllm_amd
from gpu_util import f32, log_case, t16, ti
from helpers import TOL_BF16, assert_close, random_case
from rllm_amd import ops

pytestmark = pytest.mark.gpu
TORCH = {O.BF16: torch.bfloat16, O.F16: torch.float16}

# (head_dim, q heads, kv heads, block size, kind, contexts): windows are 128
# tokens, rounds 512, head_dim classes end at 64, 96, 128, 192, 256, a group
# holds 16 heads
DECODE = [
    (128, 3, 1, 16, O.BF16, [1, 7, 8, 9, 15, 16, 17, 127, 128, 129]),
    (128, 6, 2, 16, O.F16, [511, 512, 513, 1023, 1024, 1025, 2600]),
    (96, 17, 1, 8, O.F16, [0, 130, 640]),
    (72, 33, 1, 24, O.BF16, [0, 25, 700]),
    (200, 5, 5, 40, O.F16, [1, 41, 513]),
    (256, 20, 4, 64, O.BF16, [63, 65, 2049]),
    (8, 2, 1, 32, O.BF16, [5, 33, 600]),
]


def _decode(dev, case, q, k, v, bt, sl, scale):
    D, hq, hkv, bs, kind, _ = case
    qb, kb, vb = O.encode(q, kind), O.encode(k, kind), O.encode(v, kind)
    out = ops.paged_decode(t16(qb, TORCH[kind], dev), t16(kb, TORCH[kind], dev), t16(vb, TORCH[kind], dev),
                           ti(bt, torch.int32, dev), ti(sl, torch.int32, dev), scale)
    torch.cuda.synchronize()
    return f32(out), O.paged_attention_decode(qb, kind, kb, vb, kind, bt, sl, scale, precision=1)


@pytest.mark.parametrize("case", DECODE, ids=[f"D{c[0]}-{c[1]}x{c[2]}-bs{c[3]}" for c in DECODE])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_decode_edges_vs_oracle(dev, case, sign):
    D, hq, hkv, bs, kind, lens = case
    rng = np.random.default_rng(D + hq)
    q, k, v, bt, sl = random_case(rng, len(lens), hq, hkv, D, (max(lens), max(lens)), bs=bs, neg_blocks=1)
    sl[:] = lens
    log_case(f"generic mfma decode {case} sign {sign}")
    got, ref = _decode(dev, case, q, k, v, bt, sl, sign / np.sqrt(D))
    assert_close(got, ref, TOL_BF16, f"decode {case}")
    # outputs keep the fp32 weights' precision: relative L2 within the output
    # rounding (2^-9 / 2^-12 per element, uniform) and a factor 1.5
    live = np.array(lens) > 0
    rel = np.linalg.norm(got[live] - ref[live]) / np.linalg.norm(ref[live])
    assert rel < 1.5 * (2.0 ** -9 if kind == O.BF16 else 2.0 ** -12), rel


@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("past", [True, False])
def test_decode_values_that_are_not_finite(dev, bad, past):
    # slots past the context are not read; an attended infinity or NaN reaches
    # its own row and head_dim only, as a sum over the visible keys gives it
    case = (128, 6, 2, 16, O.BF16, [40, 600])
    rng = np.random.default_rng(5)
    q, k, v, bt, sl = random_case(rng, 2, 6, 2, 128, (600, 600))
    sl[:] = [40, 600]
    pos = 40 if past else 17
    v[bt[0, pos // 16], 1, 3, pos % 16] = bad
    if past:
        k[bt[0, pos // 16], 1, 3, pos % 16] = bad
    log_case(f"generic mfma decode value {bad} past {past}")
    got, ref = _decode(dev, case, q, k, v, bt, sl, 1 / np.sqrt(128))
    assert np.array_equal(np.isfinite(got), np.isfinite(ref))
    assert np.array_equal(np.isposinf(got), np.isposinf(ref))
    ok = np.isfinite(ref)
    assert ok.all() == past
    assert (np.abs(got[ok] - ref[ok]) <= 2e-2 + 1e-2 * np.abs(ref[ok])).all()


def test_decode_repeats_bitwise_and_unsplit_agrees(dev):
    # context parts merge in order; a capture without scratch runs unsplit
    case = (96, 24, 8, 16, O.BF16, None)
    rng = np.random.default_rng(9)
    q, k, v, bt, sl = random_case(rng, 4, 24, 8, 96, (100, 3000))
    kind = O.BF16
    args = (t16(O.encode(q, kind), TORCH[kind], dev), t16(O.encode(k, kind), TORCH[kind], dev),
            t16(O.encode(v, kind), TORCH[kind], dev), ti(bt, torch.int32, dev), ti(sl, torch.int32, dev), 0.1)
    log_case("generic mfma decode repeat")
    a = ops.paged_decode(*args)
    b = ops.paged_decode(*args)
    out = torch.empty_like(a)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        ops.paged_decode(*args, out=out, validate=False)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert_close(f32(out), f32(a), TOL_BF16, "unsplit")
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


# prefill: (head_dim, q heads, kv heads, block size, kind, new tokens, cached):
# query tiles hold 128 rows (128 / G tokens), key tiles 64 keys, parts 256
PREFILL = [
    (96, 3, 3, 16, O.F16, [127, 128, 129, 1], [0, 0, 0, 0]),
    (128, 6, 2, 8, O.BF16, [42, 43, 0, 85, 1], [0, 63, 5, 65, 700]),
    (72, 5, 1, 24, O.BF16, [25, 26, 51], [0, 64, 1]),
    (200, 34, 2, 40, O.F16, [7, 8], [600, 0]),
    (256, 4, 4, 64, O.BF16, [129, 64], [63, 1000]),
    (8, 128, 1, 32, O.F16, [2, 65], [30, 0]),
]


def _prefill_case(rng, case):
    D, hq, hkv, bs, kind, new, cached = case
    new, cached = np.array(new, np.int32), np.array(cached, np.int32)
    sl = new + cached
    _, k, v, bt, _ = random_case(rng, len(new), hq, hkv, D, (int(sl.max()), int(sl.max())), bs=bs, neg_blocks=1)
    qsl = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
    q = rng.standard_normal((int(qsl[-1]), hq, D)).astype(np.float32)
    return q, k, v, bt, sl, qsl


def _prefill(dev, kind, q, k, v, bt, sl, qsl, scale):
    qb, kb, vb = O.encode(q, kind), O.encode(k, kind), O.encode(v, kind)
    out = ops.paged_prefill(t16(qb, TORCH[kind], dev), t16(kb, TORCH[kind], dev), t16(vb, TORCH[kind], dev),
                            ti(bt, torch.int32, dev), ti(sl, torch.int32, dev), ti(qsl, torch.int32, dev), scale)
    torch.cuda.synchronize()
    return f32(out), O.paged_attention_prefill(qb, kind, kb, vb, kind, bt, sl, qsl, scale, precision=1)


@pytest.mark.parametrize("case", PREFILL, ids=[f"D{c[0]}-{c[1]}x{c[2]}-bs{c[3]}" for c in PREFILL])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_prefill_edges_vs_oracle(dev, case, sign):
    D, kind = case[0], case[4]
    rng = np.random.default_rng(D + case[1])
    args = _prefill_case(rng, case)
    log_case(f"generic mfma prefill {case} sign {sign}")
    got, ref = _prefill(dev, kind, *args, sign / np.sqrt(D))
    assert_close(got, ref, TOL_BF16, f"prefill {case}")
    rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert rel < 1.5 * (2.0 ** -9 if kind == O.BF16 else 2.0 ** -12), rel


@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("cached", [0, 700])   # 700: the keys are split into parts
def test_prefill_value_that_is_not_finite_stays_in_its_rows(dev, bad, cached):
    # the value of a new token reaches the rows that see it and no earlier one
    case = (128, 6, 2, 16, O.BF16, [90], [cached])
    rng = np.random.default_rng(6)
    q, k, v, bt, sl, qsl = _prefill_case(rng, case)
    bt[bt < 0] = np.setdiff1d(np.arange(k.shape[0]), bt)[0]   # the helper's skipped block: present here
    pos = cached + 37
    v[bt[0, pos // 16], 1, 3, pos % 16] = bad
    log_case(f"generic mfma prefill value {bad} cached {cached}")
    got, ref = _prefill(dev, O.BF16, q, k, v, bt, sl, qsl, 1 / np.sqrt(128))
    ok = np.isfinite(ref)
    assert ok[:37].all() and not ok[37:, 3:, 3].any()
    assert np.array_equal(np.isfinite(got), ok) and np.array_equal(np.isposinf(got), np.isposinf(ref))
    assert (np.abs(got[ok] - ref[ok]) <= 2e-2 + 1e-2 * np.abs(ref[ok])).all()


# scores that are not finite: (head_dim, q heads, kv heads, block size, contexts)
# on the scalar routine, the matrix cores in one part and in several, and the
# stream decode's own shapes on both sides of the route
SCORES = [(36, 3, 1, 16, [40, 90]), (96, 6, 2, 16, [40, 90]), (96, 6, 2, 16, [700, 1300]),
          (128, 16, 2, 16, [40, 300]), (64, 4, 1, 16, [90, 6400]), (128, 4, 2, 16, [40, 90])]
BAD = {"k nan": np.nan, "k +inf": np.inf, "k -inf": -np.inf, "q nan": np.nan, "q inf": np.inf, "overflow": 3e19}


def _plant(bad, q_row, k_elem, fill):
    """One q or K entry that is not finite, or a product past fp32's range."""
    if bad[0] == "k":
        k_elem[...] = fill
    else:
        q_row[5] = fill
        if bad == "overflow":
            q_row[6:] = 0
            k_elem[...] = fill


def _same_but_nan(got, ref, what):
    assert np.array_equal(np.isnan(got), np.isnan(ref)), what
    ok = ~np.isnan(ref)
    assert np.isfinite(got[ok]).all() and (np.abs(got[ok] - ref[ok]) <= 2e-2 + 1e-2 * np.abs(ref[ok])).all(), what


# (the stream decode's last shape without "q nan": a row that has no score but NaN
# finds no max there and ends in zeros)
DECODE_SCORES = [(c, b) for c in SCORES for b in BAD if c != SCORES[-1] or b != "q nan"]


@pytest.mark.parametrize("case,bad", DECODE_SCORES,
                         ids=[f"D{c[0]}-{c[1]}x{c[2]}-{c[4][1]}-{b.replace(' ', '-')}" for c, b in DECODE_SCORES])
def test_decode_scores_that_are_not_finite(dev, case, bad):
    # a visible score of NaN or +inf makes its row NaN, one of -inf weighs nothing
    D, hq, hkv, bs, lens = case
    rng = np.random.default_rng(17)
    q, k, v, bt, sl = random_case(rng, 2, hq, hkv, D, (max(lens), max(lens)))
    sl[:] = lens
    _plant(bad, q[1, 0], k[bt[1, 2], 0, 5, 3:4], BAD[bad])
    log_case(f"decode scores {case} {bad}")
    got, _ = _decode(dev, (D, hq, hkv, bs, O.BF16, None), q, k, v, bt, sl, 1 / np.sqrt(D))
    qb, kb, vb = (O.encode(x, O.BF16) for x in (q, k, v))
    ref = O.paged_attention_decode(qb, O.BF16, kb, vb, O.BF16, bt, sl, 1 / np.sqrt(D), precision=0)
    assert np.isnan(ref).any() or bad == "k -inf"
    _same_but_nan(got, ref, f"{case} {bad}")


@pytest.mark.parametrize("D,hq,hkv,cached", [(36, 3, 1, 20), (128, 6, 2, 0), (128, 6, 2, 700)])
@pytest.mark.parametrize("bad", BAD, ids=[b.replace(" ", "-") for b in BAD])
def test_prefill_scores_that_are_not_finite(dev, D, hq, hkv, cached, bad):
    case = (D, hq, hkv, 16, O.BF16, [50], [cached])
    rng = np.random.default_rng(18)
    q, k, v, bt, sl, qsl = _prefill_case(rng, case)
    bt[bt < 0] = np.setdiff1d(np.arange(k.shape[0]), bt)[0]
    pos = cached + 17
    _plant(bad, q[30, 0], k[bt[0, pos // 16], 0, 5, pos % 16:pos % 16 + 1], BAD[bad])
    log_case(f"prefill scores {case} {bad}")
    got, _ = _prefill(dev, O.BF16, q, k, v, bt, sl, qsl, 1 / np.sqrt(D))
    qb, kb, vb = (O.encode(x, O.BF16) for x in (q, k, v))
    ref = O.paged_attention_prefill(qb, O.BF16, kb, vb, O.BF16, bt, sl, qsl, 1 / np.sqrt(D), precision=0)
    assert np.isnan(ref).any() and not np.isnan(ref[:17]).any() or bad == "k -inf"
    _same_but_nan(got, ref, f"{case} {bad}")


@pytest.mark.parametrize("log2w", [-16.4, -20.4, -22.4, -25.4])
@pytest.mark.parametrize("path", ["decode", "decode split", "prefill", "prefill split"])
def test_f16_tail_of_small_weights(dev, path, log2w):
    """One key outweighs a long flat tail 2^-log2w to 1 and is zero in half of the
    head_dims, which then hold the tail's share alone: about n * 2^log2w of its
    values.  Those outputs are f16 (2^-11 of their size); each weight is off by
    half of its pair's last bit at most (2^-25 - lift of the largest weight), and by
    what three fp32 roundings of the scale do to an exponent of 25 (under 2^-18) and
    the exponential and the sums (2^-20)."""
    D, hq, hkv = 96, 6, 2
    split, pre = "split" in path, "prefill" in path
    n = 2000 if split else 400
    rng = np.random.default_rng(31)
    q, k, v, bt, sl = random_case(rng, 1, hq, hkv, D, (n, n))
    # scores: 8 * 8 * scale' for the key at position 3, none for the others
    q[:], k[:] = 0, 0
    q[..., 0] = 8
    k[bt[0, 0], :, 0, 3] = 8
    scale = -log2w * np.log(2) / 64
    v[:] = np.abs(v) * 1024 + 512
    v[bt[0, 0], :, :D // 2, 3] = 0
    args = (bt, sl, scale)
    log_case(f"f16 tail {path} 2^{log2w}")
    if pre:
        qsl = np.array([0, 3], np.int32)
        got, ref = _prefill(dev, O.F16, np.repeat(q, 3, 0), k, v, bt, sl, qsl, scale)
    else:
        got, ref = _decode(dev, (D, hq, hkv, 16, O.F16, None), q, k, v, *args)
    lift = 10 if pre else 15
    rel = 2.0 ** -11 + 2.0 ** (-25 - lift - log2w) + 2.0 ** -17
    got, ref = got[..., :D // 2], ref[..., :D // 2]
    # f16's own subnormal step below 2^-14
    assert (np.abs(got - ref) <= rel * np.abs(ref) + 2.0 ** -25).all(), np.abs(got / ref - 1).max()
