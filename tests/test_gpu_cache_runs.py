"""Cache writes of long token lists (slot runs written as whole rows) against the
CPU oracle, bit-exact: prompts that start anywhere in the list and in a block,
decode tokens between them, padding, blocks past the pool, and the sizes where
groups, chunks and the choice of the kernel end."""
import numpy as np
import pytest
import torch

import oracle as O
import rllm_amd
from gpu_util import bits16, log_case, t16, t8, ti
from rllm_amd import ops
from test_gpu_rope_cache import _run as rope_run

pytestmark = pytest.mark.gpu


def _slots(rng, n, bs):
    """(slots, blocks in the pool): runs of random length at random offsets."""
    out, nb = [], 0
    while len(out) < n:
        run = int(rng.choice([1, 1, 3, 15, 16, 17, 40, 200]))
        first = int(rng.choice([0, 0, 1, 7, bs - 1]))
        out += list(range(nb * bs + first, nb * bs + first + run))
        nb = out[-1] // bs + 1 + int(rng.integers(0, 2))
    out = np.array(out[:n], np.int64)
    # blocks in any order: a run continues in an unrelated block
    perm = rng.permutation(nb + 1)
    out = perm[out // bs] * bs + out % bs
    out[rng.integers(0, n, 5)] = -1
    return out, nb - 1               # ids nb - 1 and nb lie past the pool


# (kv heads, head_dim, block size, tokens): slot runs from 393216 elements (rows below
# 256 elements: 524288), 64 of them a workgroup, 128 from 2048 tokens
SHAPES = [(8, 128, 16, 384), (8, 128, 16, 385), (8, 128, 32, 2047), (8, 128, 16, 2049), (1, 40, 48, 700),
          (3, 24, 16, 2500), (1, 8, 64, 399), (8, 128, 16, 383), (32, 128, 16, 97), (1, 264, 32, 1500),
          (2, 96, 48, 2729), (2, 96, 48, 2735), (1, 40, 48, 13111), (3, 24, 16, 7300)]


@pytest.mark.parametrize("shape", SHAPES, ids=[f"{s[0]}x{s[1]}-bs{s[2]}-n{s[3]}" for s in SHAPES])
@pytest.mark.parametrize("cache", [O.BF16, O.FP8_E4M3, O.FP8_E5M2])
def test_cache_write_runs_bit_exact(dev, shape, cache):
    hkv, d, bs, n = shape
    rng = np.random.default_rng(n + d + cache)
    sl, nb = _slots(rng, n, bs)
    nk = O.encode(rng.standard_normal((n, hkv, d)).astype(np.float32), O.BF16)
    nv = O.encode(rng.standard_normal((n, hkv, d)).astype(np.float32), O.BF16)
    args = (t16(nk, torch.bfloat16, dev), t16(nv, torch.bfloat16, dev))
    log_case(f"cache_write runs {shape} cache={cache}")
    if cache == O.BF16:
        kc = rng.integers(0, 65536, size=(nb, hkv, d, bs), dtype=np.uint16)
        vc = rng.integers(0, 65536, size=(nb, hkv, d, bs), dtype=np.uint16)
        gk, gv = t16(kc, torch.bfloat16, dev), t16(vc, torch.bfloat16, dev)
        ops.reshape_and_cache(*args, gk, gv, ti(sl, torch.int64, dev))
        torch.cuda.synchronize()
        O.cache_write(kc, vc, nk, nv, sl, bs, O.BF16, O.BF16)
        assert np.array_equal(bits16(gk), kc) and np.array_equal(bits16(gv), vc)
        return
    code = rllm_amd.DTYPE_FP8_E4M3 if cache == O.FP8_E4M3 else rllm_amd.DTYPE_FP8_E5M2
    for ks, vs, rne in ((0.25, 4.0, False), (3.7 / 448.0, 0.0117, True)):
        kc = rng.integers(0, 256, size=(nb, hkv, d, bs), dtype=np.uint8)
        vc = rng.integers(0, 256, size=(nb, hkv, d, bs), dtype=np.uint8)
        gk, gv = t8(kc, dev), t8(vc, dev)
        ops.reshape_and_cache(*args, gk, gv, ti(sl, torch.int64, dev), kv_dtype=code, k_scale=ks, v_scale=vs,
                              fp8_rounding=rllm_amd.FP8_ROUND_NEAREST_EVEN if rne
                              else rllm_amd.FP8_ROUND_TOWARD_ZERO)
        torch.cuda.synchronize()
        O.cache_write(kc, vc, nk, nv, sl, bs, O.BF16, cache, ks, vs, round_nearest=rne)
        assert np.array_equal(gk.cpu().numpy(), kc) and np.array_equal(gv.cpu().numpy(), vc)


def test_cache_write_unaligned_rows_take_the_token_kernel(dev):
    # rows two bytes past a 16-byte boundary: the same bytes
    hkv, d, bs, n = 4, 64, 16, 1600
    rng = np.random.default_rng(4)
    sl, nb = _slots(rng, n, bs)
    nk = O.encode(rng.standard_normal((n, hkv, d)).astype(np.float32), O.F16)
    buf = torch.empty(n * hkv * d + 1, dtype=torch.float16, device=dev)
    x = buf[1:].view(n, hkv, d)
    x.copy_(t16(nk, torch.float16, dev))
    kc = np.zeros((nb, hkv, d, bs), np.uint16)
    gk, gv = t16(kc, torch.float16, dev), t16(kc, torch.float16, dev)
    log_case("cache_write unaligned rows")
    ops.reshape_and_cache(x, x, gk, gv, ti(sl, torch.int64, dev))
    torch.cuda.synchronize()
    ek, ev = kc.copy(), kc.copy()
    O.cache_write(ek, ev, nk, nk, sl, bs, O.F16, O.F16)
    assert np.array_equal(bits16(gk), ek) and np.array_equal(bits16(gv), ev)


# (kv heads, head_dim, block size, tokens): whole and part groups, one token past a
# group, a block size without 16-slot groups, the widest head; each list within the
# workgroups' own groups (short) and, from 2^19 elements, 2^21 of an FP8 cache, in slot
# runs across them
ROPE_SHAPES = [(8, 128, 16, 384), (2, 64, 32, 433), (1, 16, 16, 31), (1, 96, 16, 17), (2, 80, 24, 100), (1, 512, 16, 150)]
ROPE_LONG = [(8, 128, 16, 512), (8, 64, 32, 1039), (32, 16, 16, 1025), (6, 96, 16, 913), (1, 512, 16, 1031),
             (8, 80, 24, 900), (8, 128, 16, 511), (2, 128, 16, 2100)]


@pytest.mark.parametrize("shape", ROPE_SHAPES + ROPE_LONG,
                         ids=[f"{s[0]}x{s[1]}-bs{s[2]}-n{s[3]}" for s in ROPE_SHAPES + ROPE_LONG])
@pytest.mark.parametrize("cache", [O.BF16, O.FP8_E4M3, O.FP8_E5M2])
def test_rope_cache_runs_bit_exact(dev, shape, cache):
    hkv, d, bs, n = shape
    if shape in ROPE_LONG and cache != O.BF16:
        n = 4 * n + (n & 1)
    sl, nb = _slots(np.random.default_rng(n + d), n, bs)
    rope_run(dev, n, 2 * hkv, hkv, d, nb, bs, O.BF16, cache, slots=sl, ks=0.5, vs=0.37, rne=cache == O.FP8_E5M2)


def test_rope_unaligned_cache_is_written_element_by_element(dev):
    # caches two elements past a 16-byte boundary, a list long enough for runs
    n, hkv, d, bs = 700, 8, 128, 16
    rng = np.random.default_rng(12)
    sl, nb = _slots(rng, n, bs)
    k, v = (O.encode(rng.standard_normal((n, hkv, d)).astype(np.float32), O.BF16) for _ in range(2))
    kd, vd = t16(k, torch.bfloat16, dev), t16(v, torch.bfloat16, dev)
    pos = ti(rng.integers(0, 512, n).astype(np.int32), torch.int32, dev)
    cos, sin = ops.rope_cache_tables(512, d, 10000.0, device=dev)
    size = nb * hkv * d * bs
    flat = [torch.zeros(size + 2, dtype=torch.bfloat16, device=dev) for _ in range(2)]
    odd = [f[2:].view(nb, hkv, d, bs) for f in flat]
    even = [torch.zeros((nb, hkv, d, bs), dtype=torch.bfloat16, device=dev) for _ in range(2)]
    log_case("rope, unaligned caches")
    for kc, vc in (odd, even):
        ops.rope_and_cache(None, kd, vd, kc, vc, ti(sl, torch.int64, dev), pos, cos, sin)
    torch.cuda.synchronize()
    for a, b in zip(odd, even):
        assert np.array_equal(bits16(a), bits16(b)) and b.any()
