"""Calls from two host threads at once, on two streams and on one.

The library keeps its scratch per (device, stream): the stream decode's arrival
counters and partials, the prefill's KV-split partials, the cascade's partials.
Two threads that call the decode, the chunked prefill, the mixed step and the
cascade on their own streams at the same time must therefore give the bits
that the same calls give one at a time, and the library's host state (scratch
table, occupancy cache) must stand concurrent callers.  The ctypes calls
release the GIL, so the two threads are inside the library together.

On one stream the threads share the scratch: a call of two launches (partials,
then their merge) must not have the other thread's launches between its own."""
import threading

import numpy as np
import pytest
import torch

import oracle as O
from gpu_util import RawStream, ti, t16
from rllm_amd import ops

pytestmark = pytest.mark.gpu


def _case(rng, dev):
    hq, hkv, D, bs = 32, 8, 128, 16
    # decode: 48 sequences of mixed lengths (rows cut between waves, merged
    # through the stream workspace)
    dl = rng.integers(1, 3000, size=48).astype(np.int32)
    dnb = (dl + bs - 1) // bs
    # prefill: one 512-token chunk on 1024 cached tokens (the KV-split path)
    pl = np.array([1536], np.int32)
    pnb = (pl + bs - 1) // bs
    # cascade: 32 sequences on one 16-block prefix, 8 blocks of their own
    cbt_w = 16 + 8
    pool = int(dnb.sum() + pnb.sum()) + 16 + 32 * 8 + 4
    perm = rng.permutation(pool).astype(np.int32)
    dbt = np.full((48, int(dnb.max())), -1, np.int32)
    p = 0
    for s in range(48):
        dbt[s, :dnb[s]] = perm[p:p + dnb[s]]
        p += int(dnb[s])
    pbt = perm[p:p + int(pnb[0])].reshape(1, -1).copy()
    p += int(pnb[0])
    cbt = np.empty((32, cbt_w), np.int32)
    cbt[:, :16] = perm[p:p + 16]
    cbt[:, 16:] = perm[p + 16:p + 16 + 32 * 8].reshape(32, 8)
    csl = (16 * 16 + rng.integers(1, 8 * 16, size=32)).astype(np.int32)
    cq = O.encode(rng.standard_normal((32, hq, D)).astype(np.float32), O.BF16)
    k = O.encode(rng.standard_normal((pool, hkv, D, bs)).astype(np.float32), O.BF16)
    v = O.encode(rng.standard_normal((pool, hkv, D, bs)).astype(np.float32), O.BF16)
    dq = O.encode(rng.standard_normal((48, hq, D)).astype(np.float32), O.BF16)
    pq = O.encode(rng.standard_normal((512, hq, D)).astype(np.float32), O.BF16)
    return dict(
        kc=t16(k, torch.bfloat16, dev), vc=t16(v, torch.bfloat16, dev),
        dq=t16(dq, torch.bfloat16, dev), dbt=ti(dbt, torch.int32, dev), dsl=ti(dl, torch.int32, dev),
        pq=t16(pq, torch.bfloat16, dev), pbt=ti(pbt, torch.int32, dev), psl=ti(pl, torch.int32, dev),
        qsl=ti(np.array([0, 512], np.int32), torch.int32, dev), scale=1 / np.sqrt(D),
        cq=t16(cq, torch.bfloat16, dev), cbt=ti(cbt, torch.int32, dev), csl=ti(csl, torch.int32, dev))


def _decode(c, out, stream=None):
    ops.paged_decode(c["dq"], c["kc"], c["vc"], c["dbt"], c["dsl"], c["scale"], out=out, validate=False,
                     stream=stream)


def _prefill(c, out, stream=None):
    ops.paged_prefill(c["pq"], c["kc"], c["vc"], c["pbt"], c["psl"], c["qsl"], c["scale"], out=out,
                      validate=False, stream=stream)


def _mixed(c, outs, stream=None):
    ops.paged_mixed(c["pq"], c["pbt"], c["psl"], c["qsl"], c["dq"], c["dbt"], c["dsl"], c["kc"], c["vc"],
                    c["scale"], prefill_out=outs[0], decode_out=outs[1], validate=False, stream=stream)


def _cascade(c, out, stream=None):
    ops.paged_decode_prefix(c["cq"], c["kc"], c["vc"], c["cbt"], c["csl"], c["scale"], 16, out=out,
                            validate=False, stream=stream)


def _outputs(c):
    return [torch.zeros_like(c["dq"]), torch.zeros_like(c["pq"]), torch.zeros_like(c["pq"]),
            torch.zeros_like(c["dq"]), torch.zeros_like(c["cq"])]


def _step(c, o, stream=None):
    _decode(c, o[0], stream)
    _prefill(c, o[1], stream)
    _mixed(c, (o[2], o[3]), stream)
    _cascade(c, o[4], stream)


def test_two_threads_on_two_streams_give_the_same_bits(dev, monkeypatch):
    """Decode, split prefill, the one-launch mixed step and the cascade (forced)
    on two streams from two threads, 25 rounds each."""
    monkeypatch.setenv("RLLM_CASCADE", "always")
    rng = np.random.default_rng(5150)
    c = _case(rng, dev)
    ref = _outputs(c)
    _step(c, ref)
    torch.cuda.synchronize()

    n_iter = 25
    outs = [_outputs(c) for _ in range(2)]
    errors = []
    start = threading.Barrier(2)

    def worker(i, stream):
        try:
            start.wait()
            for _ in range(n_iter):
                _step(c, outs[i], stream)
            stream.synchronize()
        except Exception as e:   # reported by the main thread
            errors.append(e)

    with RawStream() as s0, RawStream() as s1:
        torch.cuda.synchronize()
        threads = [threading.Thread(target=worker, args=(i, s)) for i, s in enumerate((s0, s1))]
        for t in threads:
            t.start()
        for t in threads:
            t.join(timeout=120)
        assert not any(t.is_alive() for t in threads), "a worker thread did not finish"
        torch.cuda.synchronize()
    assert not errors, errors
    names = ["decode", "prefill", "mixed prefill", "mixed decode", "cascade"]
    for i in range(2):
        for j, name in enumerate(names):
            assert torch.equal(outs[i][j], ref[j]), f"{name} bits differ on thread {i}"


def _two_launch_calls(rng, dev):
    """One call of every path that leaves partials for a second launch: split-K
    decode, shape-general decode (and a tuned shape that runs it), split prefill,
    shape-general split prefill, cascade."""
    c = _case(rng, dev)
    bf = torch.bfloat16

    def pool(n, hkv, d):
        return [t16(O.encode(rng.standard_normal((n, hkv, d, 16)).astype(np.float32), O.BF16), bf, dev)
                for _ in range(2)]

    def q(n, hq, d):
        return t16(O.encode(rng.standard_normal((n, hq, d)).astype(np.float32), O.BF16), bf, dev)

    gk, gv = pool(200, 8, 96)
    gq, gp = q(4, 24, 96), q(40, 24, 96)
    gbt = ti(rng.integers(0, 200, (4, 190)).astype(np.int32), torch.int32, dev)
    gsl = ti(np.array([3000, 1500, 2, 700], np.int32), torch.int32, dev)
    psl = ti(np.array([1040], np.int32), torch.int32, dev)
    pql = ti(np.array([0, 40], np.int32), torch.int32, dev)
    lk, lv = pool(300, 2, 64)
    lq = q(1, 8, 64)
    lbt = ti(rng.integers(0, 300, (1, 500)).astype(np.int32), torch.int32, dev)
    lsl = ti(np.array([7990], np.int32), torch.int32, dev)
    kw = dict(validate=False)
    return [
        (c["dq"], lambda o, s: ops.paged_decode(c["dq"], c["kc"], c["vc"], c["dbt"], c["dsl"], c["scale"],
                                                partition_size=512, out=o, stream=s, **kw)),
        (gq, lambda o, s: ops.paged_decode(gq, gk, gv, gbt, gsl, 0.1, out=o, stream=s, **kw)),
        (lq, lambda o, s: ops.paged_decode(lq, lk, lv, lbt, lsl, 0.125, out=o, stream=s, **kw)),
        (c["pq"], lambda o, s: _prefill(c, o, s)),
        (gp, lambda o, s: ops.paged_prefill(gp, gk, gv, gbt[:1], psl, pql, 0.1, out=o, stream=s, **kw)),
        (c["cq"], lambda o, s: _cascade(c, o, s)),
    ]


def test_two_threads_on_one_stream_give_the_same_bits(dev, monkeypatch):
    monkeypatch.setenv("RLLM_CASCADE", "always")
    calls = [_two_launch_calls(np.random.default_rng(61 + i), dev) for i in range(2)]
    refs = []
    for mine in calls:
        refs.append([torch.zeros_like(q) for q, _ in mine])
        for (_, call), out in zip(mine, refs[-1]):
            call(out, None)
    outs = [[torch.zeros_like(r) for r in ref] for ref in refs]
    wrong = [torch.zeros(len(ref), dtype=torch.int64, device=dev) for ref in refs]
    torch.cuda.synchronize()
    errors = []
    start = threading.Barrier(2)

    def worker(i, stream):
        try:
            start.wait()
            with torch.cuda.stream(stream):
                for _ in range(40):
                    for (_, call), out in zip(calls[i], outs[i]):
                        call(out, stream)
                    for j, out in enumerate(outs[i]):
                        wrong[i][j] += (out != refs[i][j]).any()
                        out.zero_()
        except Exception as e:   # reported by the main thread
            errors.append(e)

    with RawStream() as st:
        threads = [threading.Thread(target=worker, args=(i, st)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join(timeout=120)
        assert not any(t.is_alive() for t in threads), "a worker thread did not finish"
        torch.cuda.synchronize()
    assert not errors, errors
    for i in range(2):
        assert wrong[i].tolist() == [0] * len(refs[i]), f"calls that differ, of 40, on thread {i}"
