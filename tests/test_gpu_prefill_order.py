"""Prefill grids of more than one round of workgroups and the three ways a
workgroup finds its tile: the longest query tiles first (3 to 12 sequences, GQA 4
and 8, one to two rounds), up to 64 sequences from one lane each, more by a walk;
rows without a query beside live ones; contexts past 64 steps of 64 keys."""
import numpy as np
import pytest
import torch

import oracle as O
from gpu_util import f32, log_case, t16, ti
from helpers import TOL_BF16, assert_close
from rllm_amd import ops

pytestmark = pytest.mark.gpu


def _case(seqs, hq, hkv, d, new_max, cached, seed):
    rng = np.random.default_rng(seed)
    new = rng.integers(1, new_max, size=seqs, endpoint=True).astype(np.int32)
    if seqs > 2:
        new[rng.integers(2, seqs)] = 0                # a sequence without new tokens
    new[min(1, seqs - 1)] = new_max
    sl = new + rng.integers(0, cached, size=seqs, endpoint=True).astype(np.int32)
    if cached:
        sl[0] = new[0] + cached
    nblk = (sl + 15) // 16
    pool = int(nblk.sum()) + 1
    perm = rng.permutation(pool).astype(np.int32)
    bt = np.full((seqs, max(1, int(nblk.max()))), -1, np.int32)
    p = 0
    for s in range(seqs):
        bt[s, :nblk[s]] = perm[p:p + nblk[s]]
        p += nblk[s]
    qsl = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
    q = O.encode(rng.standard_normal((int(qsl[-1]), hq, d)).astype(np.float32), O.BF16)
    k = O.encode(rng.standard_normal((pool, hkv, d, 16)).astype(np.float32), O.BF16)
    v = O.encode(rng.standard_normal((pool, hkv, d, 16)).astype(np.float32), O.BF16)
    return q, k, v, bt, sl, qsl


# (sequences, q heads, kv heads, head_dim, longest chunk, longest cache): with 32
# kv heads 9 sequences already make more workgroups than the GPU has CUs (GQA 1:
# sequence by sequence)
CASES = [(9, 32, 32, 64, 300, 0), (16, 32, 32, 64, 520, 100), (16, 64, 8, 64, 200, 70), (3, 32, 32, 64, 1100, 5000),
         (17, 32, 32, 64, 260, 0), (64, 32, 32, 64, 40, 30), (65, 32, 32, 64, 40, 30), (1, 8, 2, 128, 65, 0)]


@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}seqs-{c[1]}x{c[2]}-D{c[3]}-{c[4]}on{c[5]}" for c in CASES])
def test_prefill_order_vs_oracle(dev, case):
    seqs, hq, hkv, d, new_max, cached = case
    q, k, v, bt, sl, qsl = _case(seqs, hq, hkv, d, new_max, cached, seqs + d)
    log_case(f"prefill order {case}")
    bf = torch.bfloat16
    out = ops.paged_prefill(t16(q, bf, dev), t16(k, bf, dev), t16(v, bf, dev), ti(bt, torch.int32, dev),
                            ti(sl, torch.int32, dev), ti(qsl, torch.int32, dev), 1 / np.sqrt(d))
    torch.cuda.synchronize()
    ref = O.paged_attention_prefill(q, O.BF16, k, v, O.BF16, bt, sl, qsl, 1 / np.sqrt(d), precision=1)
    assert_close(f32(out), ref, TOL_BF16, f"prefill order {case}")


def _lists_case(hq, hkv, d, new, cached, seed):
    rng = np.random.default_rng(seed)
    new, sl = np.array(new, np.int32), (np.array(new) + cached).astype(np.int32)
    nblk = (sl + 15) // 16
    pool = int(nblk.sum()) + 1
    perm = rng.permutation(pool).astype(np.int32)
    bt = np.full((len(new), int(nblk.max())), -1, np.int32)
    p = 0
    for s, n in enumerate(nblk):
        bt[s, :n] = perm[p:p + n]
        p += n
    qsl = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
    q, k, v = (O.encode(rng.standard_normal(shape).astype(np.float32), O.BF16)
               for shape in ((int(qsl[-1]), hq, d), (pool, hkv, d, 16), (pool, hkv, d, 16)))
    return q, k, v, bt, sl, qsl


# (q heads, kv heads, new tokens, cached tokens, workgroups): on 256 CUs the order by
# falling key counts from 273 workgroups to 512
LISTS = [(64, 16, [300, 300, 260, 130, 64, 65], [0] * 6, 336), (64, 16, [448, 320, 200, 1], [0] * 4, 272),
         (64, 16, [448, 320, 257, 1], [0, 9, 0, 700], 288), (64, 16, [512] * 4, [0] * 4, 512),
         (64, 16, [512, 512, 512, 513], [0] * 4, 528), (64, 8, [320, 200, 33, 500, 1], [64, 0, 1, 0, 63], 288),
         (64, 16, [100, 0, 130, 64, 65, 128, 1, 200, 90, 30, 70, 180], [40] * 12, 368),
         (64, 16, [300, 300, 260, 200], [5000, 0, 70, 3000], 304), (64, 16, [640, 500], [0, 0], 288),
         (64, 32, [300, 300, 260], [0, 5, 0], 288)]


@pytest.mark.parametrize("case", LISTS, ids=[f"{c[0]}x{c[1]}-{len(c[2])}seqs-{c[4]}wgs" for c in LISTS])
def test_prefill_order_of_given_lengths_vs_oracle(dev, case):
    hq, hkv, new, cached, wgs = case
    qt = 256 * hkv // hq
    assert sum((n + qt - 1) // qt for n in new) * hkv == wgs
    q, k, v, bt, sl, qsl = _lists_case(hq, hkv, 64, new, cached, wgs)
    log_case(f"prefill order {case}")
    bf = torch.bfloat16
    out = ops.paged_prefill(t16(q, bf, dev), t16(k, bf, dev), t16(v, bf, dev), ti(bt, torch.int32, dev),
                            ti(sl, torch.int32, dev), ti(qsl, torch.int32, dev), 1 / 8)
    torch.cuda.synchronize()
    ref = O.paged_attention_prefill(q, O.BF16, k, v, O.BF16, bt, sl, qsl, 1 / 8, precision=1)
    assert_close(f32(out), ref, TOL_BF16, f"prefill order {case}")


def test_context_past_the_table(dev):
    """A context far past the table is clamped to it, however long it claims to
    be: every query then sees the whole table, in the longest-first grid too."""
    q, k, v, bt, sl, qsl = _lists_case(64, 16, 64, LISTS[0][2], LISTS[0][3], 5)
    bf = torch.bfloat16
    bt = np.where(bt < 0, 0, bt).astype(np.int32)
    outs = []
    for top in (1 << 24, 2**31 - 1):
        sl[:] = top
        log_case(f"prefill order, context {top} on a table of {bt.shape[1]} blocks")
        outs.append(ops.paged_prefill(t16(q, bf, dev), t16(k, bf, dev), t16(v, bf, dev), ti(bt, torch.int32, dev),
                                      ti(sl, torch.int32, dev), ti(qsl, torch.int32, dev), 1 / np.sqrt(64),
                                      validate=False, out=torch.zeros_like(t16(q, bf, dev))))
    torch.cuda.synchronize()
    sl[:] = 1 << 24
    ref = O.paged_attention_prefill(q, O.BF16, k, v, O.BF16, bt, sl, qsl, 1 / 8, precision=1)
    assert_close(f32(outs[0]), ref, TOL_BF16, "context past the table")
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


# prefixes in 1, 4, 8 and 2 splits
@pytest.mark.parametrize("seqs,prefix,own", [(160, 16, 40), (128, 64, 16), (128, 128, 16), (32, 40, 3)])
def test_prefix_splits_match_the_plain_decode(dev, seqs, prefix, own, monkeypatch):
    rng = np.random.default_rng(seqs + prefix)
    hq, hkv, d, pool = 32, 8, 128, prefix + seqs * own
    perm = rng.permutation(pool).astype(np.int32)
    bt = np.concatenate([np.tile(perm[:prefix], (seqs, 1)), perm[prefix:].reshape(seqs, own)], axis=1)
    sl = np.full(seqs, (prefix + own) * 16, np.int32) - rng.integers(0, 16, seqs).astype(np.int32)
    g = torch.Generator(device=dev)
    g.manual_seed(seqs)
    q = torch.randn((seqs, hq, d), generator=g, device=dev, dtype=torch.bfloat16)
    k = torch.randn((pool, hkv, d, 16), generator=g, device=dev, dtype=torch.bfloat16)
    v = torch.randn((pool, hkv, d, 16), generator=g, device=dev, dtype=torch.bfloat16)
    args = (q, k, v, ti(bt, torch.int32, dev), ti(sl, torch.int32, dev), 1 / np.sqrt(d))
    log_case(f"prefix splits {seqs} x ({prefix} + {own})")
    plain = ops.paged_decode(*args)
    monkeypatch.setenv("RLLM_CASCADE", "always")
    got = ops.paged_decode_prefix(*args, prefix)
    torch.cuda.synchronize()
    assert_close(f32(got), f32(plain), TOL_BF16, "prefix splits")
