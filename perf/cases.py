"""The work this library is used for, as measurable cases.

Each case is one pass of an attention layer's work through the torch front end
(``rllm_amd.ops``), over device tensors that a serving program already holds:
decode attention (small, mixed, FP8, shared prefix, head layouts outside the
Llama ones), chunked and whole-prompt prefill, the mixed step, the cache
writes and the element-wise operators around them.  ``listed()`` names typical
sizes, ``draw()`` gives others of the same ranges; ``exact()`` computes the
same outputs with plain torch in 64 bits.

Sequence lengths belong to the case (they fix its work); block tables, slots
and values come from the seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from rllm_amd import ops
from rllm_amd._lib import DTYPE_FP8_E4M3, DTYPE_FP8_E5M2

DEVICE = "cuda"
FP8_SCALE = 0.0125            # per-tensor scale of the FP8 caches (about amax / 448 of N(0, 1) values)
ROPE_THETA = 500000.0
KV_CODE = {"same": None, "fp8_e4m3": DTYPE_FP8_E4M3, "fp8_e5m2": DTYPE_FP8_E5M2}
FP8_TORCH = {"fp8_e4m3": torch.float8_e4m3fn, "fp8_e5m2": torch.float8_e5m2}
FP8_MAX = {"fp8_e4m3": 448.0, "fp8_e5m2": 57344.0}
HALF = {"bf16": torch.bfloat16, "f16": torch.float16}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def _decode(name, batch, ctx_min, ctx_max, hq, hkv, d, bs=16, dtype="bf16", kv="same", lens=0):
    c = {"kind": "decode", "batch": batch, "ctx_min": ctx_min, "ctx_max": ctx_max, "hq": hq, "hkv": hkv,
         "d": d, "bs": bs, "dtype": dtype, "kv": kv, "lens": lens}
    return dict(c, name=name) if name else c


def _prefix(name, batch, shared, own, hq, hkv, d, dtype="bf16", kv="same"):
    c = {"kind": "prefix", "batch": batch, "shared": shared, "own": own, "hq": hq, "hkv": hkv, "d": d,
         "bs": 16, "dtype": dtype, "kv": kv}
    return dict(c, name=name) if name else c


def _prefill(name, prompts, new_min, new_max, cached, hq, hkv, d, bs=16, dtype="bf16", kv="same", lens=0):
    c = {"kind": "prefill", "prompts": prompts, "new_min": new_min, "new_max": new_max, "cached": cached,
         "hq": hq, "hkv": hkv, "d": d, "bs": bs, "dtype": dtype, "kv": kv, "lens": lens}
    return dict(c, name=name) if name else c


def _mixed(name, batch, ctx_min, ctx_max, new, cached, hq, hkv, d, dtype="bf16", kv="same", lens=0):
    c = {"kind": "mixed", "batch": batch, "ctx_min": ctx_min, "ctx_max": ctx_max, "new": new, "cached": cached,
         "hq": hq, "hkv": hkv, "d": d, "bs": 16, "dtype": dtype, "kv": kv, "lens": lens}
    return dict(c, name=name) if name else c


def _write(name, rope, runs, run_min, run_max, hq, hkv, d, bs=16, dtype="bf16", kv="same", lens=0):
    """runs sequences, each writing run_min..run_max consecutive new tokens."""
    c = {"kind": "rope" if rope else "write", "runs": runs, "run_min": run_min, "run_max": run_max, "hq": hq,
         "hkv": hkv, "d": d, "bs": bs, "dtype": dtype, "kv": kv, "lens": lens}
    return dict(c, name=name) if name else c


def _mlp(name, tokens, hidden, inner, dtype="bf16"):
    c = {"kind": "mlp", "tokens": tokens, "hidden": hidden, "inner": inner, "dtype": dtype}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: eight short chats on a 1B-size layer, latency and launches
        _decode("decode_small", 8, 512, 512, 32, 8, 64),
        # a serving batch of chats of mixed age on an 8B-size layer
        _decode("decode_mixed", 64, 128, 4096, 32, 8, 128, lens=2),
        # a full GPU of equal contexts over an FP8 cache: the largest
        _decode("decode_fp8", 256, 2048, 2048, 32, 8, 128, kv="fp8_e4m3"),
        # one system prompt shared by the batch, short turns behind it
        _prefix("decode_shared_prefix", 128, 64, 16, 32, 8, 128),
        # a model whose query heads group in threes
        _decode("decode_gqa3", 48, 64, 3000, 24, 8, 128, lens=5),
        # a scheduler's chunk of prompts whose first part is cached already
        _prefill("prefill_chunk", 8, 512, 512, 2048, 32, 8, 128),
        # fresh prompts of uneven length, f16 as in the reference's own entry points
        _prefill("prefill_prompts", 6, 100, 2048, 0, 32, 8, 128, dtype="f16", lens=7),
        # fresh prompts of a model with 96-wide heads, one kv head per query head
        _prefill("prefill_d96", 4, 100, 1024, 0, 32, 32, 96, dtype="f16", lens=8),
        # one step of a scheduler that mixes a prompt chunk into the decode batch
        _mixed("mixed_step", 64, 128, 4096, 512, 2048, 32, 8, 128, lens=2),
        # rotary embedding and cache write of a chunk of prompts
        _write("rope_write_chunk", True, 8, 512, 512, 32, 8, 128),
        # plain cache write of uneven prompts
        _write("cache_write_prompts", False, 6, 100, 1500, 32, 8, 128, lens=11),
        # the norm and the gated activation around a chunk's MLP
        _mlp("norm_and_gate", 4096, 4096, 14336),
    ]


_LLAMA_HEADS = [(32, 8), (32, 8), (16, 4), (8, 2), (4, 1), (32, 32), (32, 4)]
_OTHER_HEADS = [(24, 8), (28, 4), (40, 8), (12, 4), (48, 8), (32, 2), (16, 16), (20, 20)]
_OTHER_DIMS = [40, 64, 80, 96, 112, 128, 160, 192, 256]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _other_shape(rng):
    """Heads, head_dim and block size outside the Llama layouts."""
    while True:
        hq, hkv = rng.choice(_OTHER_HEADS + _LLAMA_HEADS[:2])
        d = rng.choice(_OTHER_DIMS)
        bs = rng.choice([16, 16, 16, 8, 32, 64])
        if not (d in (64, 128) and bs == 16 and hq // hkv in (1, 2, 4, 8)):
            return hq, hkv, d, bs


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode_other", "prefix", "prefill", "prefill", "prefill_other",
                       "mixed", "rope", "write", "write", "mlp"])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    kv = rng.choice(["same", "same", "fp8_e4m3", "fp8_e5m2"])
    e = 2 if kv == "same" else 1
    lens = rng.randrange(1 << 16)
    if kind in ("decode", "decode_other"):
        if kind == "decode":
            (hq, hkv), d, bs = rng.choice(_LLAMA_HEADS), rng.choice([64, 128, 128]), 16
            cap = 1000e6
        else:
            hq, hkv, d, bs = _other_shape(rng)
            cap = 400e6
        batch = _log_int(rng, 1, 256)
        ctx_max = _log_int(rng, 64, 32768)
        while batch * ctx_max * hkv * d * 2 * e > cap:
            if ctx_max > 2048 or batch == 1:
                ctx_max = ctx_max * 2 // 3
            else:
                batch = batch * 2 // 3
        ctx_min = rng.choice([ctx_max, max(1, ctx_max // 2), max(1, ctx_max // 32)])
        return _decode(None, batch, ctx_min, ctx_max, hq, hkv, d, bs, dtype, kv, lens)
    if kind == "prefix":
        hq, hkv = rng.choice([(32, 8), (32, 8), (16, 4), (32, 4)])
        return _prefix(None, _log_int(rng, 16, 192), _log_int(rng, 32, 256), _log_int(rng, 4, 48), hq, hkv,
                       rng.choice([64, 128, 128]), dtype, kv)
    if kind == "prefill":
        hq, hkv = rng.choice(_LLAMA_HEADS)
        d = rng.choice([64, 128, 128])
        prompts, new = _log_int(rng, 1, 8), _log_int(rng, 16, 2048)
        cached = rng.choice([0, 0, _log_int(rng, 16, 4096)])
        while 4.0 * hq * d * prompts * new * (cached + new / 2) > 150e9:
            if cached > 512:
                cached = cached * 2 // 3
            else:
                new = new * 2 // 3
        return _prefill(None, prompts, rng.choice([new, max(1, new // 20)]), new, cached, hq, hkv, d, 16, dtype, kv,
                        lens)
    if kind == "prefill_other":
        hq, hkv, d, bs = _other_shape(rng)
        prompts, new = _log_int(rng, 1, 4), _log_int(rng, 16, 1024)
        cached = rng.choice([0, 0, _log_int(rng, 16, 1024)])
        while 4.0 * hq * d * prompts * new * (cached + new / 2) > 8e9:
            if cached > 256:
                cached = cached * 2 // 3
            else:
                new = new * 2 // 3
        return _prefill(None, prompts, rng.choice([new, max(1, new // 10)]), new, cached, hq, hkv, d, bs, dtype, kv,
                        lens)
    if kind == "mixed":
        hq, hkv = rng.choice([(32, 8), (32, 8), (16, 4), (32, 4)])
        batch, ctx_max = _log_int(rng, 8, 96), _log_int(rng, 256, 4096)
        return _mixed(None, batch, rng.choice([ctx_max, max(1, ctx_max // 32)]), ctx_max, _log_int(rng, 64, 1536),
                      rng.choice([0, _log_int(rng, 64, 2048)]), hq, hkv, 128, dtype, kv, lens)
    if kind in ("rope", "write"):
        hq, hkv = rng.choice(_LLAMA_HEADS + [(24, 8)])
        d = rng.choice([64, 96, 128, 128])
        bs = rng.choice([16, 16, 16, 32])
        if rng.random() < 0.4:   # a decode step: one token per sequence
            return _write(None, kind == "rope", _log_int(rng, 1, 256), 1, 1, hq, hkv, d, bs, dtype, kv, lens)
        runs, run = _log_int(rng, 1, 8), _log_int(rng, 16, 1024)
        return _write(None, kind == "rope", runs, rng.choice([run, max(1, run // 10)]), run, hq, hkv, d, bs, dtype, kv,
                      lens)
    hidden, inner = rng.choice([(2048, 8192), (4096, 14336), (4096, 11008), (3072, 8192), (5120, 13824)])
    return _mlp(None, _log_int(rng, 1, 3000), hidden, inner, dtype)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _lens(case, n, lo, hi):
    r = np.random.default_rng([0x524C4C4D, case.get("lens", 0), n, lo, hi])
    return r.integers(lo, hi, size=n, endpoint=True).astype(np.int64)


def _gen(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed & 0x7FFFFFFF)
    return g


def _randn(g, shape, dtype):
    return torch.randn(shape, generator=g, device=DEVICE, dtype=dtype)


def _cache(case, g, num_blocks):
    """One pool [num_blocks, hkv, d, bs] of N(0, 1) values in the cache's type."""
    shape = (num_blocks, case["hkv"], case["d"], case["bs"])
    if case["kv"] == "same":
        return _randn(g, shape, HALF[case["dtype"]])
    out = torch.empty(shape, dtype=torch.uint8, device=DEVICE)
    flat = out.view(-1)
    step, top = 1 << 26, FP8_MAX[case["kv"]]
    for i in range(0, flat.numel(), step):
        n = min(step, flat.numel() - i)
        x = _randn(g, (n,), torch.float32).div_(FP8_SCALE).clamp_(-top, top)
        flat[i:i + n] = x.to(FP8_TORCH[case["kv"]]).view(torch.uint8)
    return out


def _tables(rng, lens, bs, pool_slack=1.1):
    """Scattered block ids, as a block pool hands them out: (tables, blocks in the pool)."""
    nblk = [(int(n) + bs - 1) // bs for n in lens]
    pool = int(math.ceil(pool_slack * sum(nblk))) + 1
    perm = rng.permutation(pool).astype(np.int32)
    bt = np.full((len(nblk), max(nblk)), -1, np.int32)
    p = 0
    for s, n in enumerate(nblk):
        bt[s, :n] = perm[p:p + n]
        p += n
    return bt, pool


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEVICE)


def _scale(case):
    return 1.0 / math.sqrt(case["d"])


def _kv_opts(case):
    if case["kv"] == "same":
        return {}
    return {"kv_dtype": KV_CODE[case["kv"]], "k_scale": FP8_SCALE, "v_scale": FP8_SCALE}


def _decode_lens(case):
    return _lens(case, case["batch"], case["ctx_min"], case["ctx_max"])


def _prefill_lens(case):
    new = _lens(case, case["prompts"], case["new_min"], case["new_max"])
    return new, new + case["cached"]


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    rng = np.random.default_rng([seed & 0x7FFFFFFF, 17])
    st = {"case": case}
    if kind == "mlp":
        dt = HALF[case["dtype"]]
        t, h, i = case["tokens"], case["hidden"], case["inner"]
        st["x"] = _randn(g, (t, h), dt)
        st["w"] = (1.0 + 0.1 * _randn(g, (h,), torch.float32)).to(dt)
        st["gate"], st["up"] = _randn(g, (t, i), dt), _randn(g, (t, i), dt)
        st["normed"], st["act"] = torch.empty_like(st["x"]), torch.empty_like(st["gate"])
        return st
    dt = HALF[case["dtype"]]
    hq, hkv, d, bs = case["hq"], case["hkv"], case["d"], case["bs"]
    if kind in ("rope", "write"):
        runs = _lens(case, case["runs"], case["run_min"], case["run_max"])
        # decode tokens land anywhere in their sequence's last block; prompt
        # chunks start at the front of a block, as a scheduler cuts them
        if case["run_max"] == 1:
            start = rng.integers(0, 4096, size=case["runs"])
        else:
            start = rng.integers(0, 64, size=case["runs"]) * bs
        first = start // bs
        bt, pool = _tables(rng, start + runs - first * bs, bs)
        slots, pos = [], []
        for s, n in enumerate(runs.tolist()):
            p = np.arange(start[s], start[s] + n)
            slots.append(bt[s, p // bs - first[s]].astype(np.int64) * bs + p % bs)
            pos.append(p)
        n = int(runs.sum())
        st["slots"] = _dev(np.concatenate(slots))
        st["k"], st["v"] = _randn(g, (n, hkv, d), dt), _randn(g, (n, hkv, d), dt)
        st["kc"], st["vc"] = _cache(case, g, pool), _cache(case, g, pool)
        if kind == "rope":
            st["q"] = _randn(g, (n, hq, d), dt)
            st["q_out"] = torch.empty_like(st["q"])
            st["pos"] = _dev(np.concatenate(pos).astype(np.int32))
            inv = ROPE_THETA ** (-torch.arange(0, d, 2, dtype=torch.float64) / d)
            ang = torch.arange(8192, dtype=torch.float64)[:, None] * inv[None, :]
            st["cos"], st["sin"] = ang.cos().float().to(DEVICE), ang.sin().float().to(DEVICE)
        return st
    if kind == "prefix":
        pool = case["shared"] + case["batch"] * case["own"]
        perm = rng.permutation(pool).astype(np.int32)
        bt = np.empty((case["batch"], case["shared"] + case["own"]), np.int32)
        bt[:, :case["shared"]] = perm[:case["shared"]]
        bt[:, case["shared"]:] = perm[case["shared"]:].reshape(case["batch"], case["own"])
        lens = np.full(case["batch"], bt.shape[1] * bs, np.int64)
        st["q"] = _randn(g, (case["batch"], hq, d), dt)
    elif kind == "decode":
        lens = _decode_lens(case)
        bt, pool = _tables(rng, lens, bs)
        st["q"] = _randn(g, (case["batch"], hq, d), dt)
    elif kind == "prefill":
        new, lens = _prefill_lens(case)
        bt, pool = _tables(rng, lens, bs)
        st["q"] = _randn(g, (int(new.sum()), hq, d), dt)
        st["qsl"] = _dev(np.concatenate([[0], np.cumsum(new)]).astype(np.int32))
    else:   # mixed: the prompt chunk is the last sequence of the pool's tables
        lens = np.concatenate([_decode_lens(case), [case["cached"] + case["new"]]])
        bt, pool = _tables(rng, lens, bs)
        b = case["batch"]
        st["q"] = _randn(g, (b, hq, d), dt)
        st["pq"] = _randn(g, (case["new"], hq, d), dt)
        st["qsl"] = _dev(np.array([0, case["new"]], np.int32))
        st["pbt"], st["plens"] = _dev(bt[b:]), _dev(lens[b:].astype(np.int32))
        st["pout"] = torch.empty_like(st["pq"])
        bt, lens = bt[:b], lens[:b]
    st["bt"], st["lens"] = _dev(bt), _dev(lens.astype(np.int32))
    st["kc"], st["vc"] = _cache(case, g, pool), _cache(case, g, pool)
    st["out"] = torch.empty_like(st["q"])
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "mlp":
        ops.rmsnorm(st["x"], st["w"], 1e-5, out=st["normed"])
        ops.silu_mul(st["gate"], st["up"], out=st["act"])
        return st["normed"], st["act"]
    opts = _kv_opts(case)
    if kind == "write":
        ops.reshape_and_cache(st["k"], st["v"], st["kc"], st["vc"], st["slots"], **opts)
        return st["kc"], st["vc"]
    if kind == "rope":
        ops.rope_and_cache(st["q"], st["k"], st["v"], st["kc"], st["vc"], st["slots"], st["pos"], st["cos"],
                           st["sin"], q_out=st["q_out"], **opts)
        return st["q_out"], st["kc"], st["vc"]
    scale = _scale(case)
    if kind == "decode":
        return ops.paged_decode(st["q"], st["kc"], st["vc"], st["bt"], st["lens"], scale, out=st["out"],
                                validate=False, **opts)
    if kind == "prefix":
        return ops.paged_decode_prefix(st["q"], st["kc"], st["vc"], st["bt"], st["lens"], scale, case["shared"],
                                       out=st["out"], validate=False, **opts)
    if kind == "prefill":
        return ops.paged_prefill(st["q"], st["kc"], st["vc"], st["bt"], st["lens"], st["qsl"], scale, out=st["out"],
                                 validate=False, **opts)
    return ops.paged_mixed(st["pq"], st["pbt"], st["plens"], st["qsl"], st["q"], st["bt"], st["lens"], st["kc"],
                           st["vc"], scale, prefill_out=st["pout"], decode_out=st["out"], validate=False, **opts)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _attention_work(case, new, ctx, kv_tokens):
    """new / ctx per sequence; kv_tokens: cache tokens to be read."""
    e = 2 if case["kv"] == "same" else 1
    pairs = sum(n * (c - n) + n * (n + 1) // 2 for n, c in zip(new, ctx))
    table = sum((c + case["bs"] - 1) // case["bs"] for c in ctx) * 4
    return {"bytes": int(kv_tokens * case["hkv"] * case["d"] * 2 * e + sum(new) * case["hq"] * case["d"] * 4 + table
                         + 4 * len(ctx)),
            "flops": int(4 * case["d"] * case["hq"] * pairs)}


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        t, h, i = case["tokens"], case["hidden"], case["inner"]
        return {"bytes": t * h * 4 + h * 2 + t * i * 6, "flops": t * h * 4 + t * i * 6}
    if kind in ("rope", "write"):
        n = int(_lens(case, case["runs"], case["run_min"], case["run_max"]).sum())
        e = 2 if case["kv"] == "same" else 1
        kv = case["hkv"] * case["d"] * 2
        per = kv * 2 + kv * e + 8
        if kind == "rope":
            per += case["hq"] * case["d"] * 4 + case["d"] * 4 + 4
        return {"bytes": n * per, "flops": n * (case["hq"] + case["hkv"]) * case["d"] * 3 if kind == "rope" else 0}
    if kind == "decode":
        lens = _decode_lens(case).tolist()
        return _attention_work(case, [1] * len(lens), lens, sum(lens))
    if kind == "prefix":
        n, bs = case["batch"], case["bs"]
        ctx = (case["shared"] + case["own"]) * bs
        return _attention_work(case, [1] * n, [ctx] * n, (case["shared"] + n * case["own"]) * bs)
    if kind == "prefill":
        new, ctx = _prefill_lens(case)
        return _attention_work(case, new.tolist(), ctx.tolist(), int(ctx.sum()))
    lens = _decode_lens(case).tolist()
    new, ctx = [1] * len(lens) + [case["new"]], lens + [case["cached"] + case["new"]]
    return _attention_work(case, new, ctx, sum(ctx))


def tolerance(case):
    # cache writes and the rotation are defined byte for byte
    if case["kind"] in ("rope", "write"):
        return "exact"
    # 16-bit outputs, fp32 sums; the attention weights may be 16-bit too
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 1.5e-3}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _dequant(case, cache, blocks):
    x = cache[blocks]
    if case["kv"] == "same":
        return x.double()
    return x.view(FP8_TORCH[case["kv"]]).to(torch.float32).double() * FP8_SCALE


def _attend(case, st, q, table, ctx):
    """q [n, hq, d]: the last n of ctx tokens, causal -> [n, hq, d] in 64 bits."""
    n, hq, d = q.shape
    hkv, bs = case["hkv"], case["bs"]
    g = hq // hkv
    blocks = table[:(ctx + bs - 1) // bs].long()
    k = _dequant(case, st["kc"], blocks).permute(1, 2, 0, 3).reshape(hkv, d, -1)[:, :, :ctx]
    v = _dequant(case, st["vc"], blocks).permute(1, 2, 0, 3).reshape(hkv, d, -1)[:, :, :ctx]
    out = torch.empty((n, hq, d), dtype=torch.float64, device=q.device)
    step = max(1, (1 << 26) // (hq * ctx))
    for i in range(0, n, step):
        m = min(step, n - i)
        qq = q[i:i + m].double().view(m, hkv, g, d).permute(1, 2, 0, 3).reshape(hkv, g * m, d)
        s = torch.matmul(qq, k) * _scale(case)
        if n > 1:
            last = torch.arange(ctx - n + i, ctx - n + i + m, device=q.device).repeat(g)
            s.masked_fill_(torch.arange(ctx, device=q.device)[None, None, :] > last[None, :, None], float("-inf"))
        p = torch.softmax(s, dim=-1)
        o = torch.matmul(p, v.transpose(1, 2).contiguous())
        out[i:i + m] = o.view(hkv, g, m, d).permute(2, 0, 1, 3).reshape(m, hq, d)
    return out


def _exact_write(case, st, k):
    """The two caches after the write; FP8 bytes have no 64-bit value."""
    if case["kv"] != "same":
        return None, None
    out = []
    for cache, new in ((st["kc"], k), (st["vc"], st["v"].double())):
        c = cache.double()
        blk, off = st["slots"] // case["bs"], st["slots"] % case["bs"]
        c.permute(0, 3, 1, 2)[blk, off] = new
        out.append(c)
    return tuple(out)


def _rotate(st, x):
    cos, sin = (st[t][st["pos"].long()].to(x.dtype).double()[:, None, :] for t in ("cos", "sin"))
    a, b = x.double().chunk(2, dim=-1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    if kind == "mlp":
        x = st["x"].double()
        normed = x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + float(np.float32(1e-5))) * st["w"].double()
        gate = st["gate"].double()
        return normed, gate / (1 + torch.exp(-gate)) * st["up"].double()
    if kind == "write":
        return _exact_write(case, st, st["k"].double()) if case["kv"] == "same" else None
    if kind == "rope":
        return (_rotate(st, st["q"]),) + _exact_write(case, st, _rotate(st, st["k"]))
    if kind == "prefill":
        new, ctx = _prefill_lens(case)
        parts, p = [], 0
        for s, (n, c) in enumerate(zip(new.tolist(), ctx.tolist())):
            parts.append(_attend(case, st, st["q"][p:p + n], st["bt"][s], c))
            p += n
        return torch.cat(parts)
    lens = st["lens"].tolist()
    dec = torch.cat([_attend(case, st, st["q"][s:s + 1], st["bt"][s], c) for s, c in enumerate(lens)])
    if kind != "mixed":
        return dec
    return _attend(case, st, st["pq"], st["pbt"][0], case["cached"] + case["new"]), dec
