"""Decode of the stream kernel's own shapes where few long rows (GQA 4 and 8) or
short tables (GQA 8) run the shape-general kernels instead: both sides of every
line of the rule, tables wider than any context among them, against the oracle and
the stream (an explicit workspace always takes it)."""
import numpy as np
import pytest
import torch

import oracle as O
import rllm_amd
from gpu_util import f32, log_case, t16, t8, ti
from helpers import TOL_BF16, TOL_FP8, assert_close, random_case
from rllm_amd import ops
from rllm_amd.attention import decode_workspace_size

pytestmark = pytest.mark.gpu

# (sequences, q heads, kv heads, head_dim, table blocks, cache)
CASES = [(1, 32, 8, 128, 7, O.BF16), (2, 32, 8, 128, 7, O.BF16), (1, 32, 8, 64, 9, O.BF16), (64, 32, 8, 128, 2, O.BF16),
         (65, 32, 8, 128, 2, O.BF16), (64, 32, 8, 64, 16, O.FP8_E4M3), (62, 32, 8, 64, 16, O.FP8_E4M3),
         (9, 32, 8, 128, 31, O.BF16), (9, 32, 8, 128, 33, O.BF16), (1, 4, 1, 128, 384, O.BF16), (1, 4, 1, 128, 383, O.BF16),
         (5, 8, 2, 128, 250, O.BF16), (2, 32, 4, 64, 32, O.FP8_E5M2), (2, 32, 4, 64, 33, O.BF16),
         (2, 8, 1, 128, 256, O.BF16), (3, 16, 8, 128, 7, O.BF16), (5, 8, 8, 64, 3, O.BF16),
         (128, 32, 4, 64, 3, O.BF16), (129, 32, 4, 64, 3, O.BF16), (2, 8, 1, 64, 255, O.FP8_E4M3),
         (32, 8, 1, 64, 256, O.BF16), (33, 8, 1, 64, 256, O.BF16), (24, 4, 1, 64, 384, O.BF16),
         (25, 4, 1, 64, 384, O.BF16), (1, 8, 1, 64, 16384, O.FP8_E5M2), (1, 8, 1, 64, 16385, O.FP8_E5M2)]


@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}x{c[1]}:{c[2]}-D{c[3]}-{c[4]}blk-kv{c[5]}" for c in CASES])
def test_both_routes_vs_oracle(dev, case):
    B, hq, hkv, d, maxb, kv = case
    rng = np.random.default_rng(B + maxb)
    top = min(16 * maxb, 9000)               # past that: a table wider than its contexts
    q, k, v, bt, sl = random_case(rng, B, hq, hkv, d, (1 if B > 1 else top - 3, top), max_blocks=maxb, neg_blocks=1)
    if B > 2:
        sl[0], sl[1] = top, 0
        bt[0] = rng.permutation(k.shape[0])[:maxb]
    qb = O.encode(q, O.BF16)
    bf = torch.bfloat16
    opts = {}
    if kv == O.BF16:
        kb, vb = O.encode(k, kv), O.encode(v, kv)
        kc, vc = t16(kb, bf, dev), t16(vb, bf, dev)
    else:
        kb, vb = (O.encode((x / np.float32(0.02)).astype(np.float32), kv) for x in (k, v))
        kc, vc = t8(kb, dev), t8(vb, dev)
        opts = dict(kv_dtype=rllm_amd.DTYPE_FP8_E4M3 if kv == O.FP8_E4M3 else rllm_amd.DTYPE_FP8_E5M2,
                    k_scale=0.02, v_scale=0.02)
    scale = 1 / np.sqrt(d)
    args = (t16(qb, bf, dev), kc, vc, ti(bt, torch.int32, dev), ti(sl, torch.int32, dev), scale)
    log_case(f"decode routes {case}")
    a = ops.paged_decode(*args, **opts)
    again = ops.paged_decode(*args, **opts)
    ws = torch.zeros(max(16, decode_workspace_size(B, hq, hkv, d, 16, maxb)), dtype=torch.uint8, device=dev)
    b = ops.paged_decode(*args, workspace=ws, **opts)
    torch.cuda.synchronize()
    s = 0.02 if kv != O.BF16 else 1.0
    ref = O.paged_attention_decode(qb, O.BF16, kb, vb, kv, bt, sl, scale, s, s, precision=1)
    tol = TOL_BF16 if kv == O.BF16 else TOL_FP8
    assert_close(f32(a), ref, tol, f"automatic {case}")
    assert_close(f32(b), ref, tol, f"stream {case}")
    assert torch.equal(a.view(torch.int16), again.view(torch.int16))


def test_workspace_of_a_larger_batch_serves_a_smaller(dev):
    """Whole waves per row want more scratch for 341 rows of this width than 342
    take (1023 waves against 727): a workspace sized for the larger batch still
    runs the smaller, on equal shares."""
    hq, hkv, d, maxb = 4, 1, 64, 17
    have = decode_workspace_size(342, hq, hkv, d, 16, maxb)
    assert have < decode_workspace_size(341, hq, hkv, d, 16, maxb)
    rng = np.random.default_rng(15)
    q, k, v, bt, sl = random_case(rng, 341, hq, hkv, d, (1, 272), max_blocks=maxb)
    qb = O.encode(q, O.BF16)
    kb, vb = (O.encode((x / np.float32(0.02)).astype(np.float32), O.FP8_E4M3) for x in (k, v))
    ws = torch.zeros(have, dtype=torch.uint8, device=dev)
    log_case("decode 341 rows, workspace of 342")
    out = ops.paged_decode(t16(qb, torch.bfloat16, dev), t8(kb, dev), t8(vb, dev), ti(bt, torch.int32, dev),
                           ti(sl, torch.int32, dev), 1 / 8, workspace=ws, kv_dtype=rllm_amd.DTYPE_FP8_E4M3,
                           k_scale=0.02, v_scale=0.02)
    torch.cuda.synchronize()
    ref = O.paged_attention_decode(qb, O.BF16, kb, vb, O.FP8_E4M3, bt, sl, 1 / 8, 0.02, 0.02, precision=1)
    assert_close(f32(out), ref, TOL_FP8, "workspace of a larger batch")


# (sequences, q heads, kv heads, head_dim, table blocks, cache, equal shares): whole rows
# would be 1056 waves for 1000 SIMDs' worth of equal shares; 32 waves a row
MIXED_LENGTHS = [(24, 32, 4, 128, 250, O.FP8_E4M3, 1000), (3, 16, 4, 64, 250, O.BF16, 375), (3, 16, 4, 64, 250, O.FP8_E4M3, 375)]


@pytest.mark.parametrize("case", MIXED_LENGTHS, ids=[f"{c[0]}x{c[1]}:{c[2]}-{c[4]}blk" for c in MIXED_LENGTHS])
def test_mixed_lengths_run_equal_shares(dev, case):
    """Whole waves per row serve batches of equal lengths; where rows take many
    waves, or more than the SIMDs, mixed lengths keep the equal shares, which a
    workspace of just their size leaves the call: the same bits."""
    B, hq, hkv, d, maxb, kv, shares = case
    rng = np.random.default_rng(B)
    pool = 600
    gen = torch.Generator(device=dev)
    gen.manual_seed(B)
    q = torch.randn((B, hq, d), generator=gen, device=dev, dtype=torch.bfloat16)
    if kv == O.BF16:
        kc, vc = (torch.randn((pool, hkv, d, 16), generator=gen, device=dev, dtype=torch.bfloat16) for _ in range(2))
        opts = {}
    else:
        kc, vc = (torch.randint(0, 96, (pool, hkv, d, 16), generator=gen, device=dev, dtype=torch.uint8) for _ in range(2))
        opts = dict(kv_dtype=rllm_amd.DTYPE_FP8_E4M3, k_scale=0.02, v_scale=0.02)
    bt = ti(rng.integers(0, pool, (B, maxb)).astype(np.int32), torch.int32, dev)
    sl = rng.integers(8 * maxb, 16 * maxb, B).astype(np.int32)
    size = 32 * 1024 + 2 * shares * (hq // hkv) * (d + 2) * 4
    full = decode_workspace_size(B, hq, hkv, d, 16, maxb)
    log_case(f"mixed lengths {case}")
    got = []
    for lens in (sl, np.full(B, 16 * maxb, np.int32)):
        for nbytes in (max(full, size), size):
            ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
            got.append(ops.paged_decode(q, kc, vc, bt, ti(lens, torch.int32, dev), 0.1, workspace=ws, validate=False, **opts))
    torch.cuda.synchronize()
    assert torch.equal(got[0], got[1])
    assert_close(f32(got[2]), f32(got[3]), TOL_BF16, "equal lengths")
