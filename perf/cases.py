"""The calls whose speed counts: one attention layer's cache and attention
calls and one layer's int4 projections, over the sizes a decoder meets.

A decoder calls, per layer and step, :func:`rec_amd.attend` with its new
keys and values (one token, a short turn, a prefill chunk), on the cache that
kind of layer has: the quantized cache of a full-attention layer
(``MixedQuantizedKVCache`` in its group-64 affine default, or the int8 and
uint4 formats), the bf16 storage, or a sliding layer's 513-token ring; and
it multiplies its activations by the layer's int4 matrices.  Every case is one
such call, or one layer's run of projections, eagerly from Python as a decode
loop makes them.  ``exact`` restates each from its definition in float64 (the
quantizers in float32, whose codes are the cache's own) with plain torch.
"""

from __future__ import annotations

import math

import torch

import rec_amd
from rec_amd.kvstorage import FixedKVCache, FixedSlidingKVCache, KVStorage

D = 128
SCALE = D**-0.5
WINDOW = 513
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
# (group_size, key_bits, value_bits) of the quantized formats
FORMATS = {"int8": (32, 8, 8), "uint4": (32, 4, 4), "mixed": (32, 8, 4), "affine": (64, 8, 4)}
TOKEN_BYTES = {"int8": 260, "uint4": 160, "mixed": 210, "affine": 208, "bf16": 512}  # K + V per token and KV head
# the decoder layer's matrices: hidden width, query rows, key and value rows, dense MLP width
HIDDEN, Q_ROWS, KV_ROWS, MLP = 2048, 4096, 512, 6144
HEAD_ROWS = 150144  # the lm head's rows


def _attn(name, cache, held, new, *, fmt="bf16", batch=1, q_heads=32, kv_heads=4, dtype="bf16"):
    return {"name": name, "kind": "attn", "cache": cache, "fmt": fmt, "held": held, "new": new, "batch": batch,
            "q_heads": q_heads, "kv_heads": kv_heads, "dtype": dtype}


def listed():
    return [
        # one token through a sliding-window layer: the smallest call of a decode step, and three layers in four
        _attn("ring_decode_513", "ring", 2000, 1),
        # one token over a 32K int8 cache: the headline decode step (fp16 keys, as its configuration states)
        _attn("decode_int8_32k", "quant", 32767, 1, fmt="int8", dtype="fp16"),
        # one token over a 131K uint4 cache
        _attn("decode_uint4_131k", "quant", 131071, 1, fmt="uint4", dtype="fp16"),
        # one token over the default (affine 8/4-bit) cache near the context limit, an odd count
        _attn("decode_affine_252k", "quant", 258046, 1, fmt="affine"),
        # a prompt chunk through a sliding-window layer
        _attn("ring_chunk_512", "ring", 2000, 512),
        # a short turn after a long conversation
        _attn("turn_int8_32k_20", "quant", 32768, 20, fmt="int8"),
        # an ordinary, odd prompt chunk into the default cache
        _attn("prefill_affine_4k_1000", "quant", 4097, 1000, fmt="affine"),
        # a full chunk of a long prompt: the largest call
        _attn("prefill_int8_64k_2048", "quant", 65536, 2048, fmt="int8"),
        # a prompt's keys and values written into an int8 cache at once
        {"name": "append_int8_32k", "kind": "append", "fmt": "int8", "held": 0, "new": 32768, "batch": 1,
         "kv_heads": 4, "dtype": "bf16"},
        # a decode step's projections of one layer: q, k and v stacked, o, gate and up stacked, down
        {"name": "proj_1row", "kind": "proj", "rows": 1},
        # the same for a short turn (or a batch of sequences)
        {"name": "proj_24rows", "kind": "proj", "rows": 24},
        # the same for a prefill chunk
        {"name": "proj_2000rows", "kind": "proj", "rows": 2000},
    ]


def _log_int(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(hi, max(lo, n))


def draw(rng):
    kind = rng.choice(["decode", "decode", "ring", "turn", "prefill", "append", "proj", "proj", "head"])
    if kind == "head":  # the lm head: one row per sequence of a decode step
        return {"kind": "head", "rows": rng.randint(1, 32)}
    if kind == "proj":
        return {"kind": "proj", "rows": _log_int(rng, 1, 2048)}
    fmt = rng.choice(["int8", "uint4", "mixed", "affine", "affine"])
    if kind == "append":
        return {"kind": "append", "fmt": fmt, "held": rng.randint(0, 4000), "new": _log_int(rng, 1, 65536),
                "batch": rng.choice([1, 1, 2]), "kv_heads": rng.choice([1, 4, 8]),
                "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    q_heads, kv_heads = rng.choice([(32, 4), (32, 4), (8, 1), (16, 4), (32, 8)])
    heads = {"q_heads": q_heads, "kv_heads": kv_heads}
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "ring":
        case = _attn("", "ring", _log_int(rng, 1, 8000), rng.choice([1, _log_int(rng, 2, 1024)]), **heads)
    elif kind == "decode":
        batch = rng.choice([1, 1, 2, 4])
        held = _log_int(rng, 512, 262000 // batch)
        cache, dt = rng.choice([("quant", dtype), ("quant", "fp32"), ("store", "bf16")])
        case = _attn("", cache, held, 1, fmt=fmt if cache == "quant" else "bf16", batch=batch, dtype=dt, **heads)
    elif kind == "turn":
        case = _attn("", "quant", _log_int(rng, 512, 131072), rng.randint(2, 48), fmt=fmt, dtype=dtype, **heads)
    else:
        cache = rng.choice(["quant", "quant", "store"])
        new, held = _log_int(rng, 64, 1500), rng.choice([0, _log_int(rng, 256, 50000)])
        case = _attn("", cache, held, new, fmt=fmt if cache == "quant" else "bf16", dtype=dtype if cache == "quant"
                     else "bf16", **heads)
    del case["name"]
    return case


# ------------------------------------------------------------------ inputs --


def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt) % (1 << 62))
    return g


def _rows(g, B, H, T, dtype, fmt):
    """N(0, 1) keys or values with outlier channels (1% of them at 8 times the
    size; for the 4-bit format 5% heavy-tailed ones), the shape real caches show."""
    x = torch.randn((B, H, T, D), generator=g, device="cuda", dtype=torch.float32)
    n = 6 if fmt in ("uint4", "mixed") else 1
    idx = torch.randperm(D, generator=g, device="cuda")[:n]
    if n == 1:
        x[..., idx] *= 8.0
    else:
        t = torch.randn((B, H, T, n, 3), generator=g, device="cuda").square_().sum(-1).div_(3.0).clamp_min_(1e-2)
        x[..., idx] = x[..., idx] / t.sqrt_()
    return x.to(dtype)


def _attn_inputs(case, seed):
    B, H, dt = case["batch"], case["kv_heads"], DTYPES[case["dtype"]]
    kv_dt = dt if case["cache"] == "quant" else torch.bfloat16
    new, held, fmt = case["new"], case["held"], case["fmt"]
    old = tuple(_rows(_gen(seed, s), B, H, held, kv_dt, fmt) for s in (1, 2)) if held else (None, None)
    k, v = (_rows(_gen(seed, s), B, H, new, kv_dt, fmt) for s in (3, 4))
    q = torch.randn((B, case["q_heads"], new, D), generator=_gen(seed, 5), device="cuda").to(dt)
    sinks = torch.randn((case["q_heads"],), generator=_gen(seed, 6), device="cuda")
    return old, k, v, q, sinks


def _weights(seed, salt, N, K):
    """An MLX-layout affine 4-bit matrix whose scales and biases are those of
    quantized normal weights: a range of about 16 steps around zero."""
    g = _gen(seed, salt)
    w = torch.randint(-(2**31), 2**31, (N, K // 8), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
    s = (torch.rand((N, K // 64), generator=g, device="cuda") * 0.01 + 0.002).to(torch.bfloat16)
    b = (s.float() * (-7.5 + torch.randn((N, K // 64), generator=g, device="cuda"))).to(torch.bfloat16)
    return w, s, b


def _activations(seed, salt, M, K):
    g = _gen(seed, salt)
    return torch.randn((M, K), generator=g, device="cuda").to(torch.bfloat16)


def _layer(seed):
    return {"qkv": [_weights(seed, 10 + i, n, HIDDEN) for i, n in enumerate((Q_ROWS, KV_ROWS, KV_ROWS))],
            "o": [_weights(seed, 20, HIDDEN, Q_ROWS)],
            "mlp": [_weights(seed, 30 + i, MLP, HIDDEN) for i in range(2)],
            "down": [_weights(seed, 40, HIDDEN, MLP)]}


def _layer_inputs(case, seed):
    M = case["rows"]
    return {"qkv": _activations(seed, 51, M, HIDDEN), "o": _activations(seed, 52, M, Q_ROWS),
            "mlp": _activations(seed, 53, M, HIDDEN), "down": _activations(seed, 54, M, MLP)}


def _cache(case, tokens):
    fmt, B, H = case["fmt"], case["batch"], case["kv_heads"]
    if case.get("cache", "quant") == "quant":
        group, kb, vb = FORMATS[fmt]
        return rec_amd.QuantizedKVCache(group, kb, vb, max_tokens=tokens)
    if case["cache"] == "store":
        return FixedKVCache(KVStorage(1, tokens, H, batch=B), 0)
    return FixedSlidingKVCache(max_sequence_tokens=1 << 18, num_kv_heads=H, head_dim=D, window_size=WINDOW, batch=B)


def prepare(case, seed):
    if case["kind"] == "proj":
        mats = {k: rec_amd.Q4Matrix.stack(v) for k, v in _layer(seed).items()}
        return {"kind": "proj", "mats": mats, "x": _layer_inputs(case, seed)}
    if case["kind"] == "head":
        return {"kind": "head", "mat": rec_amd.Q4Matrix(*_weights(seed, 60, HEAD_ROWS, HIDDEN)),
                "x": _activations(seed, 61, case["rows"], HIDDEN)}
    cache = _cache(case, case["held"] + case["new"])
    if case["kind"] == "append":
        case = dict(case, cache="quant", q_heads=case["kv_heads"])
        old, k, v, _, _ = _attn_inputs(case, seed)
        if case["held"]:
            cache.update_and_fetch(*old)
        return {"kind": "append", "cache": cache, "k": k, "v": v}
    old, k, v, q, sinks = _attn_inputs(case, seed)
    if case["held"]:
        cache.update_and_fetch(*old)
    return {"kind": case["cache"], "cache": cache, "q": q, "k": k, "v": v, "sinks": sinks,
            "mask": None if case["new"] == 1 else "causal"}


# --------------------------------------------------------------- the calls --


def run(state):
    kind = state["kind"]
    if kind == "proj":
        m, x = state["mats"], state["x"]
        q, k, v = rec_amd.q4_gemv_parts(x["qkv"], m["qkv"])
        o = rec_amd.q4_gemv(x["o"], m["o"])
        gate, up = rec_amd.q4_gemv_parts(x["mlp"], m["mlp"])
        down = rec_amd.q4_gemv(x["down"], m["down"])
        return {"q": q, "k": k, "v": v, "o": o, "gate": gate, "up": up, "down": down}
    if kind == "head":
        return {"logits": rec_amd.q4_gemv(state["x"], state["mat"], torch.float32)}
    cache, k, v = state["cache"], state["k"], state["v"]
    n = k.shape[2]
    if kind == "append":
        keys, values = cache.update_and_fetch(k, v)
        cache.trim(n)  # the next pass writes the same positions again
        return {"k": list(keys[:3]), "v": list(values[:3])}
    out = rec_amd.attend(state["q"], k, v, cache, SCALE, state["mask"], state["sinks"])
    # roll back, so that the next pass is the same step again (a ring goes on: its oldest tokens are gone)
    if kind == "quant":
        cache.trim(n)
        return {"out": out, "k": list(cache.keys), "v": list(cache.values)}
    if kind == "store":
        cache.offset -= n
        return {"out": out}
    return {"out": out, "ring": list(cache.state)}


def work(case):
    if case["kind"] in ("proj", "head"):
        M = case["rows"]
        shapes = [(HEAD_ROWS, HIDDEN)] if case["kind"] == "head" else [
            (Q_ROWS + 2 * KV_ROWS, HIDDEN), (HIDDEN, Q_ROWS), (2 * MLP, HIDDEN), (HIDDEN, MLP)]
        out = 4 if case["kind"] == "head" else 2
        return {"bytes": sum(N * K * 0.5625 + M * K * 2 + M * N * out for N, K in shapes),
                "flops": sum(2.0 * M * N * K for N, K in shapes)}
    B, H, new, held = case["batch"], case["kv_heads"], case["new"], case["held"]
    width = 4 if case["dtype"] == "fp32" else 2
    if case["kind"] == "append":
        return {"bytes": B * H * new * (2 * D * width + TOKEN_BYTES[case["fmt"]]), "flops": 0}
    if case["cache"] == "ring":
        held = min(held, WINDOW)
    per, Hq = TOKEN_BYTES[case["fmt"]], case["q_heads"]
    # cache read, new rows read and stored, queries read, outputs written
    data = B * H * ((held + new) * per + new * 2 * D * width + new * per) + 2 * B * Hq * new * D * width
    if case["cache"] == "ring":
        pairs = sum(min(WINDOW, held + i + 1) for i in range(new))
    else:
        pairs = new * held + new * (new + 1) // 2
    return {"bytes": data, "flops": 4.0 * B * Hq * D * pairs}


def tolerance(case):
    if case["kind"] == "append":
        return "exact"
    # about four times the error measured against exact()
    if case["kind"] == "head":
        return {"rel": 1e-5}  # float32 logits of exact products, sums in another order
    if case["kind"] == "proj" or case["dtype"] == "bf16":
        return {"rel": 7e-3}  # bf16 results: one rounding each
    if case["fmt"] == "affine":
        return {"rel": 5e-3}  # values with a large common bias that cancels in the output
    if case["new"] > 1:
        return {"rel": 4e-3}  # fp16 chunks: probabilities rounded once to fp16
    return {"rel": 1.2e-3}


# ------------------------------------------------------ float64 references --


def _over(x, n):
    """x / n, correctly rounded (a Python divisor would become a multiplication)."""
    return x / torch.full_like(x, n)


def _quant_i8(x):
    """(codes, scale) of the symmetric int8 format."""
    x = x.float()
    s = _over(x.abs().amax(-1, keepdim=True), 127.0).clamp(max=65504.0).half().float()
    return torch.where(s > 0, torch.round(x / torch.where(s > 0, s, 1.0)).clamp(-127, 127), 0.0), s


def _deq_i8(x):
    q, s = _quant_i8(x)
    return q.double() * s.double()


def _deq_u4(x):
    g = x.float().reshape(*x.shape[:-1], D // 32, 32)
    mn, mx = g.amin(-1, keepdim=True).clamp(max=0.0), g.amax(-1, keepdim=True).clamp(min=0.0)
    s = _over(mx - mn, 15.0).clamp(max=65504.0).half().float()
    d = torch.where(s > 0, s, 1.0)
    z = torch.round(-mn / d).clamp(0, 15)
    q = (torch.round(g / d) + z).clamp(0, 15)
    return torch.where(s > 0, (q - z).double() * s.double(), 0.0).reshape(x.shape)


def _deq_affine(x, bits):
    n = float(2**bits - 1)
    g = x.float().reshape(*x.shape[:-1], D // 64, 64)
    mn, mx = g.amin(-1, keepdim=True), g.amax(-1, keepdim=True).clamp(min=0.0)
    s = _over(mx - mn, n).clamp(min=1e-7)
    side = mn.abs() > mx.abs()
    s = torch.where(side, s, -s)
    edge = torch.where(side, mn, mx)

    def away(t):  # round half away from zero
        return torch.sign(t) * torch.floor(t.abs() + 0.5)

    qe = away(edge / s)
    zero = qe == 0
    s = torch.where(zero, s, edge / torch.where(zero, 1.0, qe))
    b = torch.where(zero, 0.0, edge)
    q = away((g - b) / s).clamp(0, n)
    meta = torch.float16 if x.dtype == torch.float16 else torch.bfloat16
    return (q.double() * s.to(meta).double() + b.to(meta).double()).reshape(x.shape)


def _deq(x, fmt, is_v):
    if fmt == "bf16":
        return x.double()
    if fmt == "affine":
        return _deq_affine(x, 4 if is_v else 8)
    if fmt == "uint4" or (fmt == "mixed" and is_v):
        return _deq_u4(x)
    return _deq_i8(x)


def _exact_attn(case, seed):
    old, k, v, q, sinks = _attn_inputs(case, seed)
    held, new, fmt = case["held"], case["new"], case["fmt"]
    B, H, Hq = case["batch"], case["kv_heads"], case["q_heads"]
    if case["cache"] == "ring" and held > WINDOW:
        old, held = tuple(t[:, :, held - WINDOW:] for t in old), WINDOW
    sk = sinks.double() if new == 1 and case["cache"] == "quant" else sinks.to(q.dtype).double()
    out = torch.empty((B, Hq, new, D), dtype=torch.float64, device="cuda")
    qpos = torch.arange(held, held + new, device="cuda")[:, None]
    kpos = torch.arange(held + new, device="cuda")[None]
    keep = kpos <= qpos
    if case["cache"] == "ring":
        keep &= kpos > qpos - WINDOW
    for b in range(B):
        for h in range(H):
            kk, vv = (torch.cat([_deq(t[b, h], fmt, is_v) for t in ts if t is not None])
                      for is_v, ts in ((False, (old[0], k)), (True, (old[1], v))))
            if new > 1 and fmt in ("uint4", "mixed", "affine"):  # chunks see 4-bit and affine values in the query dtype
                vv = vv.float().to(q.dtype).double()
                if fmt != "mixed":
                    kk = kk.float().to(q.dtype).double()
            for i in range(h * (Hq // H), (h + 1) * (Hq // H)):
                s = (q[b, i].double() @ kk.T).mul_(SCALE)
                s.masked_fill_(~keep, -math.inf)
                top = torch.maximum(s.amax(-1, keepdim=True), sk[i])
                p = s.sub_(top).exp_()
                out[b, i] = (p @ vv) / (p.sum(-1, keepdim=True) + (sk[i] - top).exp())
                del s, p
    return out


def _matmul(x, mat):
    w, s, b = mat
    N, K = w.shape[0], w.shape[1] * 8
    shifts = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    out = []
    for r in range(0, N, 8192):
        q = ((w[r:r + 8192].unsqueeze(-1) >> shifts) & 15).reshape(-1, K // 64, 64).double()
        W = (q * s[r:r + 8192].double().unsqueeze(-1) + b[r:r + 8192].double().unsqueeze(-1)).reshape(-1, K)
        out.append(x.double() @ W.T)
    return torch.cat(out, 1)


def exact(case, seed):
    if case["kind"] == "head":
        return {"logits": _matmul(_activations(seed, 61, case["rows"], HIDDEN), _weights(seed, 60, HEAD_ROWS, HIDDEN))}
    if case["kind"] == "proj":
        mats, x = _layer(seed), _layer_inputs(case, seed)
        y = {k: [_matmul(x[k], m) for m in v] for k, v in mats.items()}
        (q, k, v), (o,), (gate, up), (down,) = y["qkv"], y["o"], y["mlp"], y["down"]
        return {"q": q, "k": k, "v": v, "o": o, "gate": gate, "up": up, "down": down}
    if case["kind"] == "append":
        return None  # bytes in the cache's own order: compared as they are
    out = {"out": _exact_attn(case, seed)}
    if case["cache"] == "quant":
        out.update(k=None, v=None)
    elif case["cache"] == "ring":
        out.update(ring=None)
    return out
