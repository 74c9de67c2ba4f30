"""Measured workloads of the attention path: decode steps and layer prefills.

One pass is one layer's call through the C ABI (include/molot_amd/attn_hip.h),
as a serving loop makes it: buffers, RoPE tables, norm weights and block
tables are laid out beforehand, the call is enqueued on the current stream.

A case is a dict of plain values:
  path    "decode" (one sequence, token-major cache), "paged" (a batch of
          sequences over 16-row pages), "prefill" (a prompt into a token-major
          cache), "prefill_paged" (a prompt into one sequence's pages)
  nq, nkv, d   query heads, KV heads, head dim
  kv      "f32", "bf16" or "q8" cache rows
  pos     decode: position of the new token (= rows cached before it)
  batch, lo, hi   paged: sequences, their contexts spread over [lo, hi]
  m, n0   prefill: prompt rows, rows cached before them
  window  sliding window (0: none);  norms  the layer's q/k/v norms
  theta   RoPE base;  sigma  standard deviation of the cached values
"""
import ctypes
import math

import torch

from molot_amd import attn
from molot_amd import lib as _lib

PAGE = 16
EPS = 1e-6
KV = {"f32": attn.KV_F32, "bf16": attn.KV_BF16, "q8": attn.KV_Q8}

# A dense 32q/8kv layer, its 64-query variant, and gemma4's two layer kinds
# (sliding window with 256-wide heads, global with 512-wide heads).
DENSE = dict(nq=32, nkv=8, d=128, theta=500000.0, window=0, norms=False, sigma=1.0)
WIDE_Q = dict(DENSE, nq=64, sigma=0.5)
LOCAL = dict(nq=8, nkv=4, d=256, theta=10000.0, window=1024, norms=True, sigma=1.0)
GLOBAL = dict(nq=8, nkv=2, d=512, theta=1000000.0, window=0, norms=True, sigma=1.0)


def listed():
    return [
        # The first tokens of a chat: latency and launches, hardly any cache.
        dict(DENSE, name="decode_first", path="decode", kv="f32", pos=300),
        # One stream at 16k context, the reference's cache type: the headline step.
        dict(DENSE, name="decode_16k", path="decode", kv="f32", pos=16384),
        # A sliding-window layer late in a long chat: a short stream behind the layer's norms.
        dict(LOCAL, name="decode_window", path="decode", kv="f32", pos=32768),
        # One very long document over a bf16 cache.
        dict(WIDE_Q, name="decode_131k_bf16", path="decode", kv="bf16", pos=131072),
        # A global 512-wide layer at 32k context over the small cache type.
        dict(GLOBAL, name="decode_d512_q8", path="decode", kv="q8", pos=32768),
        # A full continuous batch: 64 sequences of very different contexts.
        dict(DENSE, name="paged_64_bf16", path="paged", kv="bf16", batch=64, lo=512, hi=8192),
        # A small batch of ragged contexts over the small cache type.
        dict(DENSE, name="paged_13_q8", path="paged", kv="q8", batch=13, lo=1, hi=2999),
        # A short chat turn: an odd number of prompt rows into a sequence's pages.
        dict(DENSE, name="prefill_short_bf16", path="prefill_paged", kv="bf16", m=77, n0=0),
        # A fresh 2048-token prompt over the reference's cache type.
        dict(DENSE, name="prefill_2k", path="prefill", kv="f32", m=2048, n0=0),
        # The next 512 tokens of a long document: a chunk behind 16k cached rows.
        dict(DENSE, name="prefill_chunk_bf16", path="prefill", kv="bf16", m=512, n0=16384),
        # A 2048-token prompt through a sliding-window layer with its norms.
        dict(LOCAL, name="prefill_window", path="prefill", kv="f32", m=2048, n0=0),
        # A ragged prompt through a global 512-wide layer.
        dict(GLOBAL, name="prefill_d512", path="prefill", kv="f32", m=1999, n0=0),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """A case of the same ranges: contexts, prompts and batches spread over
    their logarithm, every layer kind and cache type, also 64-wide heads."""
    layer = dict(rng.choice([DENSE, WIDE_Q, LOCAL, GLOBAL, dict(DENSE, d=64)]))
    layer["norms"] = rng.random() < 0.5
    layer["kv"] = rng.choice(["f32", "bf16", "q8"])
    path = rng.choice(["decode", "decode", "paged", "prefill", "prefill_paged"])
    if path == "decode":
        hi = 131072 if layer["kv"] != "f32" else 65536
        return dict(layer, path=path, pos=_log_int(rng, 1, hi))
    if path == "paged":
        if layer["kv"] == "f32":
            layer["kv"] = "bf16"
        hi = _log_int(rng, 33, 8191 if layer["nq"] * layer["d"] < 8192 else 4095)
        return dict(layer, path=path, batch=_log_int(rng, 1, 64), lo=max(1, hi // rng.randint(2, 20)),
                    hi=hi)
    m = _log_int(rng, 2, 2047 if layer["nq"] < 64 else 1023)
    n0 = 0 if rng.random() < 0.5 else _log_int(rng, 1, 16384 * 128 // (m + 128))
    return dict(layer, path=path, m=m, n0=n0)


# --- shapes -----------------------------------------------------------------


def _contexts(case):
    """Rows cached per sequence before the new token: evenly spread over
    [lo, hi], dealt in a fixed mixed order (a batch is not sorted)."""
    b, lo, hi = case["batch"], case["lo"], case["hi"]
    at = [lo + (hi - lo) * i // max(1, b - 1) for i in range(b)]
    step = next(s for s in range(max(2, (5 * b) // 8), 10 * b + 2) if math.gcd(s, b) == 1)
    return [at[(i * step) % b] for i in range(b)]


def _first(pos, window):
    return max(0, pos - window + 1) if window > 0 else 0


def _row_bytes(case):
    d = case["d"]
    return {"f32": 4 * d, "bf16": 2 * d, "q8": d + 4}[case["kv"]]


def work(case):
    """Attended cache rows read once; q read, o written and q rotated; the new
    k/v rows read as fp32 and stored.  4*d flops per (q head, query, key)."""
    nq, nkv, d, w = case["nq"], case["nkv"], case["d"], case["window"]
    rb = _row_bytes(case)
    if case["path"] in ("decode", "paged"):
        ctx = [case["pos"]] if case["path"] == "decode" else _contexts(case)
        rows = sum(n - _first(n, w) for n in ctx)  # cached rows read
        new, pairs = len(ctx), rows + len(ctx)
    else:
        m, n0 = case["m"], case["n0"]
        rows = n0 - min(n0, _first(n0, w))
        new = m
        pairs = sum(n0 + i + 1 - _first(n0 + i, w) for i in range(m))
    io = new * (3 * nq * d * 4 + 2 * nkv * (4 * d + rb))
    return {"bytes": 2 * nkv * rows * rb + io, "flops": 4 * d * nq * pairs}


def tolerance(case):
    # o against 64 bits, and between two runs that sum in another order: up to 4.3e-7 (2-norm)
    # and 2.5e-6 (largest) seen.  Stored 16-bit rows may round the other way where the fp32 value
    # differs in its last bit, and a Q8 code may move by one there.
    if case["kv"] == "f32":
        return {"rel": 2e-6, "max": 2e-5}
    if case["kv"] == "bf16":
        return {"rel": 5e-5, "max": 8e-3}
    return {"rel": 5e-5, "max": 1e-3, "differ": 5e-3}


# --- inputs -----------------------------------------------------------------


def _quantize(x):
    """Q8 rows of x[..., d]: fp32 scale absmax/127 (1 for a zero row), codes."""
    s = x.abs().amax(-1) / 127.0
    s = torch.where(s > 0, s, torch.ones_like(s))
    return torch.clamp(torch.round(x / s[..., None]), -127, 127).to(torch.int8), s


def _cache(case, g, rows):
    """A token-major cache of `rows` random rows [rows][nkv][d]."""
    nkv, d = case["nkv"], case["d"]
    x = torch.randn(rows, nkv, d, device="cuda", generator=g) * case["sigma"]
    if case["kv"] == "f32":
        return x.view(rows, nkv * d)
    if case["kv"] == "bf16":
        return x.to(torch.bfloat16).view(rows, nkv * d)
    out = torch.zeros(rows, attn.q8_row_bytes(nkv, d), dtype=torch.uint8, device="cuda")
    codes, s = _quantize(x)
    out[:, :nkv * d] = codes.view(rows, nkv * d).view(torch.uint8)
    out[:, nkv * d:nkv * d + 4 * nkv] = s.contiguous().view(torch.uint8)
    return out


def _pool(case, g, blocks):
    """A pool of `blocks` random pages [blocks][nkv][PAGE][d]."""
    nkv, d = case["nkv"], case["d"]
    x = torch.randn(blocks, nkv, PAGE, d, device="cuda", generator=g) * case["sigma"]
    if case["kv"] == "f32":
        return x.view(blocks, -1)
    if case["kv"] == "bf16":
        return x.to(torch.bfloat16).view(blocks, -1)
    codes, s = _quantize(x)
    return torch.cat([codes.view(blocks, -1).view(torch.uint8),
                      s.contiguous().view(blocks, -1).view(torch.uint8)], 1)


def _p(t):
    return ctypes.c_void_p(None if t is None else t.data_ptr())


def prepare(case, seed):
    L = _lib.load()
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    nq, nkv, d = case["nq"], case["nkv"], case["d"]
    kvd, scale, w = KV[case["kv"]], 1.0 / math.sqrt(d), case["window"]
    path = case["path"]
    ctx = {"decode": lambda: [case["pos"]], "paged": lambda: _contexts(case)}.get(path)
    new = len(ctx()) if ctx else case["m"]
    q = torch.randn(new, nq, d, device="cuda", generator=g)
    kn = torch.randn(new, nkv, d, device="cuda", generator=g)
    vn = torch.randn(new, nkv, d, device="cuda", generator=g) * case["sigma"]
    inv = attn.rope_inv_freq(case["theta"], d).cuda()
    wq = wk = None
    if case["norms"]:
        wq, wk = (1 + 0.2 * torch.randn(2, d, device="cuda", generator=g)).unbind(0)
    o = torch.empty(new, nq, d, device="cuda")
    s = dict(q=q, kn=kn, vn=vn, inv=inv, wq=wq, wk=wk, o=o)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    i32 = dict(dtype=torch.int32, device="cuda")
    if path in ("decode", "prefill"):
        n0 = case["pos"] if path == "decode" else case["n0"]
        s["K"], s["V"] = (_cache(case, g, n0 + new) for _ in range(2))
        s["stored"] = (s["K"][n0:], s["V"][n0:])
    else:
        ctx = ctx() if ctx else [case["n0"]]
        grow = 1 if path == "paged" else new
        need = [(n + grow + PAGE - 1) // PAGE for n in ctx]
        perm = torch.randperm(sum(need) + 7, device="cuda", generator=g).to(torch.int32)
        width, at = max(need), 0
        table = torch.zeros(len(ctx), width, **i32)
        for b, k in enumerate(need):
            table[b, :k] = perm[at:at + k]
            at += k
        s["K"], s["V"] = (_pool(case, g, sum(need) + 7) for _ in range(2))
        s["stored"] = (s["K"], s["V"])
        s["table"], s["lens"] = table, torch.tensor([n + 1 for n in ctx], **i32)
        s["ctx"] = ctx
    P = {k: _p(s[k]) for k in ("q", "kn", "vn", "K", "V", "o", "inv", "wq", "wk")}
    head = (P["q"], P["kn"], P["vn"], P["K"], P["V"], P["o"])
    norm = (P["wq"], P["wk"], 1 if case["norms"] else 0, EPS) if case["norms"] else ()
    tail = (P["inv"], scale, w, kvd, stream)
    if path == "decode":
        fn = L.molot_hip_decode_step_norm if norm else L.molot_hip_decode_step
        args = head + (nq, nkv, d, n0, n0) + norm + tail
    elif path == "paged":
        fn = L.molot_hip_decode_step_paged_norm if norm else L.molot_hip_decode_step_paged
        args = (head + (_p(s["table"]), _p(s["lens"]), _p(None), len(ctx), width, max(ctx) + 1, nq,
                        nkv, d, PAGE) + norm + tail)
    else:
        norm = norm or (_p(None), _p(None), 0, EPS)
        if path == "prefill":
            fn, args = L.molot_hip_prefill_step, head + (nq, nkv, d, new, n0, n0) + norm + tail
        else:
            fn = L.molot_hip_prefill_step_paged
            args = head + (_p(s["table"]), width, PAGE, nq, nkv, d, new, ctx[0], ctx[0]) + norm + tail
    s["fn"], s["args"] = fn, args
    s["out"] = {"o": o, "q": q, "k": s["stored"][0], "v": s["stored"][1]}
    return s


def run(state):
    status = state["fn"](*state["args"])
    if status:
        raise _lib.MolotHipError(status, "attention step")
    return state["out"]


# --- the same in 64 bits ----------------------------------------------------


def _rope(x, pos, inv):
    """x[n][heads][d] rotated at pos[n]: pairs (i, i + d/2), the angle the
    fp32 product pos * inv_freq (the interface fixes it)."""
    ang = (pos.float()[:, None] * inv).double()[:, None, :]
    c, s = ang.cos(), ang.sin()
    a, b = x.chunk(2, -1)
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _rms(x, dims, w=None):
    y = x / torch.sqrt(x.square().mean(dims, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _stored(case, x):
    """Row values as the cache holds them, and as 64-bit numbers."""
    if case["kv"] == "f32":
        return x
    if case["kv"] == "bf16":
        return x.float().to(torch.bfloat16).double()
    codes, s = _quantize(x.float())
    return codes.double() * s.double()[..., None]


def _rows(case, state, name, b, n):
    """Rows 0..n-1 of sequence b as 64-bit numbers [n][nkv][d]."""
    nkv, d, x = case["nkv"], case["d"], state[name]
    if case["path"] in ("decode", "prefill"):
        if case["kv"] != "q8":
            return x[:n].view(n, nkv, d).double()
        codes = x[:n, :nkv * d].contiguous().view(torch.int8).view(n, nkv, d)
        s = x[:n, nkv * d:nkv * d + 4 * nkv].contiguous().view(torch.float32)
        return codes.double() * s.double()[..., None]
    k = (n + PAGE - 1) // PAGE
    x = x[state["table"][b, :k].long()]
    if case["kv"] == "q8":
        cut = nkv * PAGE * d
        codes = x[:, :cut].contiguous().view(torch.int8).view(k, nkv, PAGE, d)
        s = x[:, cut:].contiguous().view(torch.float32).view(k, nkv, PAGE)
        x = codes.double() * s.double()[..., None]
    else:
        x = x.view(k, nkv, PAGE, d).double()
    return x.permute(0, 2, 1, 3).reshape(k * PAGE, nkv, d)[:n]


def _attend(case, q, K, V, pos0):
    """Causal attention of q[m][nq][d] at pos0.. over K, V[n][nkv][d]."""
    nq, nkv, d, w = case["nq"], case["nkv"], case["d"], case["window"]
    m, n, G = q.shape[0], K.shape[0], nq // nkv
    out = torch.empty_like(q)
    keys = torch.arange(n, device=q.device)
    for i in range(0, m, 256):
        pos = pos0 + torch.arange(i, min(m, i + 256), device=q.device)
        dead = keys[None, :] > pos[:, None]
        if w > 0:
            dead |= keys[None, :] < (pos - w + 1)[:, None]
        for h in range(nq):
            s = q[i:i + 256, h] @ K[:, h // G].T / math.sqrt(d)
            out[i:i + 256, h] = s.masked_fill_(dead, -math.inf).softmax(-1) @ V[:, h // G]
    return out


def exact(case, seed):
    s = prepare(case, seed)
    q, k, v = (s[x].double() for x in ("q", "kn", "vn"))
    new = q.shape[0]
    if case["norms"]:
        q, k, v = _rms(q, -1, s["wq"]), _rms(k, -1, s["wk"]), _rms(v, (-2, -1))
    if case["path"] == "decode" or case["path"].startswith("prefill"):
        ctx = [case["pos"] if case["path"] == "decode" else case["n0"]]
        pos = ctx[0] + torch.arange(new, device="cuda")
    else:
        ctx = s["ctx"]
        pos = torch.tensor(ctx, device="cuda")
    q, k = _rope(q, pos, s["inv"]), _rope(k, pos, s["inv"])
    k, v = _stored(case, k), _stored(case, v)
    if len(ctx) == 1:
        K, V = (torch.cat([_rows(case, s, x, 0, ctx[0]), y]) for x, y in (("K", k), ("V", v)))
        o = _attend(case, q, K, V, ctx[0])
    else:
        o = torch.empty_like(q)
        for b, n in enumerate(ctx):
            K, V = (torch.cat([_rows(case, s, x, b, n), y[b:b + 1]]) for x, y in (("K", k), ("V", v)))
            o[b:b + 1] = _attend(case, q[b:b + 1], K, V, n)
    plain = case["path"] in ("decode", "prefill") and case["kv"] != "q8"
    return {"o": o, "q": q, "k": k.view(new, -1) if plain else None,
            "v": v.view(new, -1) if plain else None}
