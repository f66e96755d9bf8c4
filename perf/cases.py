"""The workloads the framework's speed is measured on.

Every case is a dict of plain values; ``prepare`` makes what a serving or
training program holds before the call (pools, block tables over a shuffled
pool, queries, new rows, one engine kept for the whole program, asynchronous on
torch's current stream), ``run`` makes one pass through the public engine API
(``pagedattentionmetal_amd.PagedAttentionEngine``), ``exact`` gives the same
result in 64 bits with plain torch.

Kinds of case:
  decode    paged decode of a ragged batch (f32, f16 or e4m3 pools, optional window)
  step      one sequence's decode step: append the new token, then decode it
  mixed     a continuous-batching step: prefill chunks, decode rows, their append
  prefill   a causal prompt chunk after cached context
  fused     a whole prompt: append of its rows and causal prefill in one call
  append    quantise-on-append of a prompt's rows into e4m3 pools
  backward  gradients of full attention over one sequence

K and V are N(0, 0.5^2) for f16 and f32 pools; e4m3 pools hold N(0, 1) rows with
1% of the entries eight times larger, one scale per block (amax / 448).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from pagedattentionmetal_amd import PagedAttentionEngine, PagedLayerSpec

F32, F16, E4M3 = 0, 1, 2
TORCH = {F32: torch.float32, F16: torch.float16, E4M3: torch.uint8}
ELEM = {F32: 4, F16: 2, E4M3: 1}
IO = {F32: 4, F16: 2, E4M3: 2}

# (query heads, kv heads): the configurations' 8/8, 32/8 and 64/8, and the head
# layouts of the test sweeps
HEADS = [(8, 8), (16, 4), (32, 8), (64, 8), (16, 16), (32, 32), (8, 1), (12, 4), (32, 2)]


# ------------------------------------------------------------------ the cases


def listed():
    return [
        # a handful of short chats on an f32 multi-head layer: a few MB of KV, launch and latency bound
        dict(name="decode_f32_b4", kind="decode", dtype=F32, heads=8, kv_heads=8, dim=128, block=16, batch=4,
             len_lo=17, len_hi=200, window=0, draw=1),
        # a serving batch on a grouped-query f16 layer: 0.5 GB of KV, HBM bound
        dict(name="decode_f16_b64", kind="decode", dtype=F16, heads=32, kv_heads=8, dim=128, block=16, batch=64,
             len_lo=128, len_hi=4096, window=0, draw=2),
        # a large batch over quantised pools with a long tail of lengths
        dict(name="decode_e4m3_b256", kind="decode", dtype=E4M3, heads=32, kv_heads=8, dim=128, block=16, batch=256,
             len_lo=16, len_hi=8192, window=0, draw=4),
        # long contexts behind a 4096-token window, 64 query heads
        dict(name="decode_f16_window", kind="decode", dtype=F16, heads=64, kv_heads=8, dim=128, block=16, batch=32,
             len_lo=8192, len_hi=32768, window=4096, draw=5),
        # a multi-head (ungrouped) f16 layer of head size 64, a medium batch
        dict(name="decode_f16_mha", kind="decode", dtype=F16, heads=16, kv_heads=16, dim=64, block=16, batch=24,
             len_lo=100, len_hi=3000, window=0, draw=6),
        # one interactive user: append one token, decode it over 4 K of context
        dict(name="step_f16_b1", kind="step", dtype=F16, heads=32, kv_heads=8, dim=128, block=16, length=4133),
        # a continuous-batching step: 8 chunks of 512 tokens and 56 decode rows
        dict(name="mixed_f16", kind="mixed", dtype=F16, heads=32, kv_heads=8, dim=128, block=16, chunks=8, chunk=512,
             ctx_hi=3584, decodes=56, len_lo=256, len_hi=4096, draw=3),
        # a new 4 K prompt on an f16 grouped-query layer
        dict(name="fused_f16_4096", kind="fused", dtype=F16, heads=32, kv_heads=8, dim=128, block=16, tokens=4096),
        # a prompt's second chunk on the f32 multi-head layer, ragged length and offset
        dict(name="prefill_f32_chunk", kind="prefill", dtype=F32, heads=8, kv_heads=8, dim=128, block=16, tokens=777,
             offset=391),
        # a 2 K prompt written into quantised pools
        dict(name="append_e4m3", kind="append", dtype=E4M3, heads=32, kv_heads=8, dim=128, block=16, tokens=2000,
             offset=37),
        # training: the backward of a 2 K sequence on the f16 grouped-query layer
        dict(name="backward_f16_2048", kind="backward", dtype=F16, heads=32, kv_heads=8, dim=128, block=16,
             tokens=2048),
        # training in f32 at head size 64, a short ragged sequence
        dict(name="backward_f32_600", kind="backward", dtype=F32, heads=8, kv_heads=2, dim=64, block=16, tokens=600),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_once(rng):
    kind = rng.choice(["decode", "decode", "decode", "step", "mixed", "prefill", "prefill", "fused", "append",
                       "backward", "backward"])
    heads, kv = rng.choice(HEADS)
    block = rng.choice([16, 16, 16, 8, 32, 64])
    c = dict(kind=kind, heads=heads, kv_heads=kv, block=block)
    if kind == "decode":
        hi = _log_int(rng, 64, 8192)
        c.update(dtype=rng.choice([F32, F16, F16, E4M3, E4M3]), dim=rng.choice([64, 96, 128, 128, 256]),
                 batch=_log_int(rng, 1, 256), len_lo=rng.randint(1, max(1, hi // 4)), len_hi=hi,
                 window=rng.choice([0, 0, rng.randint(64, 4096)]), draw=rng.randrange(1 << 20))
    elif kind == "step":
        c.update(dtype=rng.choice([F32, F16]), dim=rng.choice([64, 128]), length=_log_int(rng, 32, 16384))
    elif kind == "mixed":
        lo = rng.randint(1, 1024)
        c.update(dtype=rng.choice([F16, F16, E4M3]), dim=rng.choice([64, 128]), chunks=rng.randint(1, 8),
                 chunk=_log_int(rng, 32, 512), ctx_hi=rng.randint(0, 3584), decodes=rng.randint(1, 64), len_lo=lo,
                 len_hi=rng.randint(lo, 4096), draw=rng.randrange(1 << 20))
    elif kind == "prefill":
        c.update(dtype=rng.choice([F32, F16, E4M3]), dim=rng.choice([64, 96, 128]), tokens=_log_int(rng, 17, 2048),
                 offset=rng.choice([0, rng.randint(1, 2048)]))
    elif kind == "fused":
        c.update(dtype=rng.choice([F32, F16, F16]), dim=rng.choice([64, 128]), tokens=_log_int(rng, 17, 4096))
    elif kind == "append":
        c.update(dtype=E4M3, dim=rng.choice([64, 96, 128]), tokens=_log_int(rng, 1, 4096), offset=rng.randint(0, 4096))
    else:
        c.update(dtype=rng.choice([F32, F16]), dim=rng.choice([64, 128, 128]), tokens=_log_int(rng, 33, 2048))
    return c


def draw(rng):
    while True:
        c = _draw_once(rng)
        w = work(c)
        narrow = c["dtype"] == F16 and c["dim"] == 128 or c["kind"] in ("decode", "step", "append")
        # no more than the largest listed cases of the kind and type
        flops = {"backward": 2e11, "mixed": 1.9e11}.get(c["kind"], 1.5e11) if narrow else 6e9
        if w["bytes"] <= 6e8 and w["flops"] <= flops:
            return c


# ------------------------------------------------------------------ sizes


def _lens(c):
    """The row lengths of a batch: fixed by the case, whatever the inputs' seed."""
    r = np.random.default_rng(c["draw"])
    lo, hi, n = c["len_lo"], c["len_hi"], c["batch"]
    if c["dtype"] == E4M3 and hi >= 16 * lo:  # lognormal around the geometric mean
        x = np.exp(r.normal(math.log(math.sqrt(lo * hi)), 1.0, n))
        return np.clip(np.round(x), lo, hi).astype(np.int64)
    return r.integers(lo, hi + 1, n).astype(np.int64)


def _mixed_lens(c):
    """(cached tokens, new tokens) of a mixed step's sequences."""
    r = np.random.default_rng(c["draw"])
    ctx = np.concatenate([r.integers(0, c["ctx_hi"] + 1, c["chunks"]),
                          r.integers(c["len_lo"], c["len_hi"] + 1, c["decodes"]) - 1])
    new = np.concatenate([np.full(c["chunks"], c["chunk"]), np.ones(c["decodes"])])
    return ctx.astype(np.int32), new.astype(np.int32)


def work(c):
    H, K, d, dt = c["heads"], c["kv_heads"], c["dim"], c["dtype"]
    kv_tok = 2 * K * d * ELEM[dt]      # a cached token's K and V
    in_tok = 2 * K * d * IO[dt]        # a new token's K and V as they come in
    q_tok = H * d * IO[dt]
    scale = 4 / c["block"] if dt == E4M3 else 0
    if c["kind"] in ("decode", "step"):
        L = _lens(c) if c["kind"] == "decode" else np.array([c["length"]], np.int64)
        w = c.get("window", 0)
        eff = np.minimum(L, w) if w else L
        n = len(L)
        b = eff.sum() * (kv_tok + scale) + 2 * n * q_tok + (eff // c["block"]).sum() * 4
        if c["kind"] == "step":
            b += in_tok + kv_tok
        return {"bytes": float(b), "flops": float(4 * d * H * eff.sum())}
    if c["kind"] == "mixed":
        ctx, new = (x.astype(np.int64) for x in _mixed_lens(c))
        pairs = (new * ctx + new * (new + 1) // 2).sum()
        b = ctx.sum() * (kv_tok + scale) + new.sum() * (in_tok + kv_tok + 2 * q_tok)
        return {"bytes": float(b), "flops": float(4 * d * H * pairs)}
    T, off = c["tokens"], c.get("offset", 0)
    if c["kind"] == "append":
        return {"bytes": float(T * (in_tok + kv_tok)), "flops": 0.0}
    if c["kind"] == "backward":  # q, dO in, dQ out; K, V in, dK, dV out; m and l
        return {"bytes": float(T * (3 * q_tok + 2 * kv_tok + 8 * H)), "flops": float(10 * d * H * T * T)}
    b = (off + T) * kv_tok + T * 2 * q_tok
    if c["kind"] == "fused":
        b = T * (in_tok + kv_tok + 2 * q_tok)
    return {"bytes": float(b), "flops": float(4 * d * H * (T * off + T * (T + 1) // 2))}


# ------------------------------------------------------------------ inputs

_ENGINE = None


def _engine():
    """The program's one engine, set up as a serving loop does."""
    global _ENGINE
    if _ENGINE is None:
        _ENGINE = PagedAttentionEngine()
        _ENGINE.set_graceful_degradation(False)
        _ENGINE.set_gpu_timing(False)
        _ENGINE.synchronous = False
    _ENGINE.set_stream(torch.cuda.current_stream())
    return _ENGINE


def _tables(rng, lens, bs):
    """Block tables of the sequences over a shuffled pool, zero padded, and the pool's blocks."""
    n = (np.asarray(lens, np.int64) + bs - 1) // bs
    pool = int(n.sum()) + 8
    perm = rng.permutation(pool).astype(np.int32)
    bt = np.zeros((len(n), max(1, int(n.max()))), np.int32)
    at = 0
    for i, k in enumerate(n):
        bt[i, :k] = perm[at:at + k]
        at += int(k)
    return bt, pool


def _normal(gen, shape, dtype, std):
    return torch.empty(shape, device="cuda", dtype=dtype).normal_(0.0, std, generator=gen)


def _outliers(gen, x):
    return x * (1 + 7 * (torch.rand(x.shape, device="cuda", generator=gen) < 0.01)).to(x.dtype)


def _pool(gen, c, blocks):
    """One pool's contents and, for e4m3, the blocks' scales."""
    shape = (blocks, c["block"], c["kv_heads"], c["dim"])
    if c["dtype"] != E4M3:
        return _normal(gen, shape, TORCH[c["dtype"]], 0.5), None
    x = _outliers(gen, _normal(gen, shape, torch.float16, 1.0))
    s = (x.abs().amax((1, 2, 3)).float() / 448).half()
    q = (x.float() / s.float()[:, None, None, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    return q.view(torch.uint8), s


def _inputs(c, seed):
    """Everything the case is given, from the seed alone, without the framework's code."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    kind, H, K, d, bs = c["kind"], c["heads"], c["kv_heads"], c["dim"], c["block"]
    io = torch.float32 if c["dtype"] == F32 else torch.float16
    if kind == "decode":
        lens = _lens(c)
        rows = len(lens)
    elif kind == "step":
        lens, rows = np.array([c["length"]], np.int64), 1
    elif kind == "mixed":
        ctx, new = _mixed_lens(c)
        lens, rows = (ctx + new).astype(np.int64), int(new.sum())
    else:
        rows = c["tokens"]
        lens = np.array([c.get("offset", 0) + rows], np.int64)
    bt, blocks = _tables(rng, lens, bs)
    s = {"bt": torch.from_numpy(bt).cuda(), "lens": torch.from_numpy(lens.astype(np.int32)).cuda(), "rows": rows,
         "blocks": blocks}
    s["q"] = _normal(gen, (rows, H, d), io, 1.0)
    if kind in ("fused", "append"):
        for n in ("k", "v"):
            s[n] = torch.zeros((blocks, bs, K, d), dtype=TORCH[c["dtype"]], device="cuda")
            s[n + "s"] = torch.zeros(blocks, dtype=torch.float16, device="cuda") if c["dtype"] == E4M3 else None
    else:
        for n in ("k", "v"):
            s[n], s[n + "s"] = _pool(gen, c, blocks)
    if kind in ("step", "mixed", "fused", "append"):
        new = 1 if kind == "step" else rows
        for n in ("nk", "nv"):
            x = _normal(gen, (new, K, d), io, 1.0 if c["dtype"] == E4M3 else 0.5)
            s[n] = _outliers(gen, x) if c["dtype"] == E4M3 else x
    if kind == "mixed":
        s["ctx"], s["new"] = _mixed_lens(c)
    if kind == "backward":
        s["do"] = _normal(gen, (rows, H, d), io, 1.0)
        k = _rows64(c, s, "k", 0, rows)
        s["m"] = torch.empty((rows, H), dtype=torch.float32, device="cuda")
        s["l"] = torch.empty_like(s["m"])
        for h in range(H):  # the forward's row maxima and sums
            x = (s["q"][:, h].double() @ k[:, h * K // H].t().contiguous()) / math.sqrt(d)
            mx = x.amax(1).float()
            s["m"][:, h] = mx
            s["l"][:, h] = (x - mx.double()[:, None]).exp().sum(1).float()
    return s


def prepare(c, seed):
    s = _inputs(c, seed)
    s["case"] = c
    s["engine"] = _engine()
    s["layer"] = PagedLayerSpec(c["dim"], c["heads"], c["kv_heads"], c["block"], c["dtype"], c.get("window", 0))
    s["out"] = torch.empty_like(s["q"])
    if c["kind"] == "backward":
        s["dk"], s["dv"] = torch.zeros_like(s["k"]), torch.zeros_like(s["v"])
    return s


# ------------------------------------------------------------------ one pass


def run(s):
    e, c, kind, lay = s["engine"], s["case"], s["case"]["kind"], s["layer"]
    if kind == "decode":
        e.decode(s["q"], s["k"], s["v"], s["bt"], s["lens"], s["out"], s["rows"], s["bt"].shape[1], lay,
                 k_scale=s["ks"], v_scale=s["vs"])
        return s["out"]
    if kind == "step":
        e.append_to_cache(s["nk"], s["nv"], s["k"], s["v"], s["bt"], c["length"] - 1, 1, lay)
        e.decode(s["q"], s["k"], s["v"], s["bt"], s["lens"], s["out"], 1, s["bt"].shape[1], lay)
        return [s["out"], s["k"], s["v"]]
    if kind == "mixed":
        e.mixed_step(s["q"], s["out"], s["k"], s["v"], s["bt"], s["ctx"], s["new"], lay, new_keys=s["nk"],
                     new_values=s["nv"], k_scale=s["ks"], v_scale=s["vs"])
        return [s["out"], s["k"], s["v"]] + ([s["ks"], s["vs"]] if c["dtype"] == E4M3 else [])
    if kind == "prefill":
        e.prefill(s["q"], s["k"], s["v"], s["bt"], s["out"], c["tokens"], lay, causal=True, q_offset=c["offset"],
                  k_scale=s["ks"], v_scale=s["vs"])
        return s["out"]
    if kind == "fused":
        e.fused_prefill(s["q"], s["nk"], s["nv"], s["bt"], s["k"], s["v"], s["out"], c["tokens"], lay, causal=True)
        return [s["out"], s["k"], s["v"]]
    if kind == "append":
        e.append_to_cache(s["nk"], s["nv"], s["k"], s["v"], s["bt"], c["offset"], c["tokens"], lay, k_scale=s["ks"],
                          v_scale=s["vs"])
        return [s["k"], s["v"], s["ks"], s["vs"]]
    # the gradient pools are accumulated into: a training step clears them first
    s["dk"].zero_()
    s["dv"].zero_()
    e.backward(s["q"], s["k"], s["v"], s["bt"], s["do"], s["m"], s["l"], s["out"], s["dk"], s["dv"], c["tokens"], lay)
    return [s["out"], s["dk"], s["dv"]]


# ------------------------------------------------------------------ tolerances


def tolerance(c):
    """Largest difference of another correct implementation at the same precision,
    about four times what these paths show against ``exact``: f16 results carry
    their rounding (2^-11) and that of f16 probabilities (2.9e-4, largest 5.6e-3);
    f32 results the order of their sums (8.8e-7, largest 7.6e-6).  Codes and
    scales of an append are bit-exact."""
    if c["kind"] == "append":
        return "exact"
    if c["dtype"] == F32:
        return {"rel": 4e-6, "max": 4e-5}
    return {"rel": 1.2e-3, "max": 2e-2}


# ------------------------------------------------------------------ 64 bits


def _rows64(c, s, n, seq, length, lo=0):
    """Tokens lo .. length - 1 of a sequence's K or V as float64 [tokens, kv heads, d]."""
    bs = c["block"]
    t = torch.arange(lo, length, device="cuda")
    phys = s["bt"][seq].long()[t // bs]
    x = s[n][phys, t % bs]
    if c["dtype"] == E4M3:  # an element is code * scale rounded to binary16
        x = x.view(torch.float8_e4m3fn).half() * s[n + "s"][phys][:, None, None]
    return x.double()


def _attend64(q, k, v, first):
    """Causal attention of rows q [T, H, d] at positions first .. first + T - 1 over k, v [n, K, d]."""
    T, H, d = q.shape
    K = k.shape[1]
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    pos = torch.arange(T, device="cuda")[:, None] + first
    hide = torch.arange(k.shape[0], device="cuda")[None, :] > pos
    for h in range(H):
        g = h * K // H
        x = (q[:, h].double() @ k[:, g].t().contiguous()) / math.sqrt(d)
        x = torch.softmax(x.masked_fill(hide, -math.inf), 1)
        out[:, h] = x @ v[:, g].contiguous()
    return out


def _slots(c, s, seq, lo, hi):
    t = torch.arange(lo, hi, device="cuda")
    return s["bt"][seq].long()[t // c["block"]], t % c["block"]


def _decode64(c, s):
    """One query row per sequence over its (windowed) context."""
    H, K, d = c["heads"], c["kv_heads"], c["dim"]
    lens = s["lens"].tolist()
    out = torch.empty((len(lens), H, d), dtype=torch.float64, device="cuda")
    for i, L in enumerate(lens):
        lo = max(0, L - c["window"]) if c.get("window") else 0
        k, v = _rows64(c, s, "k", i, L, lo), _rows64(c, s, "v", i, L, lo)
        q = s["q"][i].double().view(K, H // K, d)
        x = torch.softmax((q @ k.permute(1, 2, 0).contiguous()) / math.sqrt(d), 2)
        out[i] = (x @ v.transpose(0, 1).contiguous()).view(H, d)
    return out


def _backward64(c, s):
    H, K, d, T = c["heads"], c["kv_heads"], c["dim"], c["tokens"]
    k, v = _rows64(c, s, "k", 0, T), _rows64(c, s, "v", 0, T)
    dq = torch.empty((T, H, d), dtype=torch.float64, device="cuda")
    dk, dv = torch.zeros_like(k), torch.zeros_like(v)
    for h in range(H):
        g = h * K // H
        kh, vh, q, do = k[:, g].contiguous(), v[:, g].contiguous(), s["q"][:, h].double(), s["do"][:, h].double()
        p = ((q @ kh.t().contiguous()) / math.sqrt(d) - s["m"][:, h].double()[:, None]).exp()
        p /= s["l"][:, h].double()[:, None]
        dp = do @ vh.t().contiguous()
        ds = p * (dp - (p * dp).sum(1, keepdim=True)) / math.sqrt(d)
        dq[:, h] = ds @ kh
        dk[:, g] += ds.t().contiguous() @ q
        dv[:, g] += p.t().contiguous() @ do
    out = [dq]
    at = _slots(c, s, 0, 0, T)
    for x in (dk, dv):
        pool = torch.zeros((s["blocks"], c["block"], K, d), dtype=torch.float64, device="cuda")
        pool[at] = x
        out.append(pool)
    return out


def exact(c, seed):
    kind, s = c["kind"], _inputs(c, seed)
    if kind == "append":
        # scales: the largest magnitude a block receives over 448; codes are whole numbers
        T, off, bs = c["tokens"], c["offset"], c["block"]
        phys = s["bt"][0].long()[(torch.arange(T, device="cuda") + off) // bs]
        out = [None, None]
        for n in ("nk", "nv"):
            x = torch.zeros(s["blocks"], dtype=torch.float64, device="cuda")
            x.scatter_reduce_(0, phys, s[n].double().abs().amax((1, 2)) / 448, "amax")
            out.append(x)
        return out
    if kind == "backward":
        return _backward64(c, s)
    if kind == "decode":
        return _decode64(c, s)
    if kind == "prefill":
        n = c["offset"] + c["tokens"]
        return _attend64(s["q"], _rows64(c, s, "k", 0, n), _rows64(c, s, "v", 0, n), c["offset"])
    if kind in ("step", "fused"):
        lo, hi = (c["length"] - 1, c["length"]) if kind == "step" else (0, c["tokens"])
        at = _slots(c, s, 0, lo, hi)
        for n in ("k", "v"):
            s[n][at] = s["n" + n]
        out = _decode64(c, s) if kind == "step" else _attend64(s["q"], s["nk"].double(), s["nv"].double(), 0)
        return [out, s["k"].double(), s["v"].double()]
    if c["dtype"] == E4M3:  # the step quantises its rows by the sticky-scale rule: no 64-bit form of that
        return None
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    row = 0
    for i, (cl, n) in enumerate(zip(s["ctx"].tolist(), s["new"].tolist())):
        at = _slots(c, s, i, cl, cl + n)
        for x in ("k", "v"):
            s[x][at] = s["n" + x][row:row + n]
        k, v = _rows64(c, s, "k", i, cl + n), _rows64(c, s, "v", i, cl + n)
        out[row:row + n] = _attend64(s["q"][row:row + n], k, v, cl)
        row += n
    return [out, None, None]
