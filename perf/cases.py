"""The work a serving engine has this library do, as measurable cases.

Every case is one call (or the usual pair of calls) of the public binding
(``mgprims.Prims``) at sizes of this repository's configurations and tests:
the 30B-class shapes (d = 5120, ffn 25600, 40 query / 8 kv heads of 128, V =
201088) and the checkpoint's (d = 6656, ffn 19968, 32 / 2 heads, V = 202048),
from one decode token to a 4096-token prompt. Inputs are seeded draws of the
distributions the benchmark uses; outputs are returned whole.

``listed()`` names the cases, ``draw(rng)`` draws more of the same ranges;
``prepare`` makes a case's inputs, ``run`` is one pass, ``work`` its minimum
bytes and operations, ``tolerance`` how far another correct implementation of
the same precision may be off, and ``exact`` the result in 64 bits, by plain
torch.
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "muse-glimmer-intel-serve_amd"))

import mgprims as M  # noqa: E402

DEV = "cuda:0"
HD = 128  # head dimension of both configurations
EPS = 1e-6
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
SCALE = 1.0 / math.sqrt(HD)
QK_SCALE = 3.87
THETA = 1e6

_prims = None


def prims():
    """One context for the process, as a program keeps it."""
    global _prims
    if _prims is None:
        _prims = M.Prims(0)
    return _prims


def listed():
    return [
        # the norm between two blocks of one decode step: a launch and its latency
        {"name": "norm_decode_1", "kind": "norm", "tokens": 1, "dim": 5120, "dtype": "bf16"},
        # the MLP's gating of a prompt of ragged length
        {"name": "swiglu_1733", "kind": "swiglu", "tokens": 1733, "ffn": 25600, "dtype": "bf16"},
        # everything around RoPE of a prompt, appended to the KV ring
        {"name": "qk_rope_kv_2000", "kind": "qk", "tokens": 2000, "heads": 40, "kv": 8, "pos0": 0},
        # the score rows of a prompt's last chunk: 1000 queries over 4000 keys
        {"name": "softmax_1000x4000", "kind": "softmax", "heads": 40, "q": 1000, "k": 4000, "pos0": 3000,
         "window": 0, "cap": 0.0},
        # attention of a whole prompt: the largest call
        {"name": "prefill_4096", "kind": "prefill", "tokens": 4096, "heads": 40, "kv": 8, "pos0": 0, "window": 0},
        # attention of a short chunk (a follow-up message, a block to verify) behind a long context
        {"name": "prefill_chunk_100", "kind": "prefill", "tokens": 100, "heads": 32, "kv": 2, "pos0": 9000,
         "window": 0},
        # one decode token at the longest context
        {"name": "decode_131072", "kind": "decode", "heads": 40, "kv": 8, "keys": 131072},
        # one decode token in an ordinary conversation
        {"name": "decode_1500", "kind": "decode", "heads": 32, "kv": 2, "keys": 1500},
        # a quantized projection at decode, one user
        {"name": "gemv_b1", "kind": "gemv", "rows": 25600, "in": 5120, "batch": 1},
        # the same for a batch of users, the down projection's shape
        {"name": "gemv_b6", "kind": "gemv", "rows": 6656, "in": 19968, "batch": 6},
        # output tail, top-64 and the sampler's distribution for a batch of 8
        {"name": "vocab_8", "kind": "vocab", "rows": 8, "V": 201088, "K": 64, "top_p": 0.95},
        # the sampler without a top-k cut, for a batch of 64
        {"name": "sampler_64", "kind": "sample", "rows": 64, "V": 201088, "top_p": 0.95, "min_p": 0.0},
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["norm", "swiglu", "qk", "softmax", "prefill", "prefill", "decode", "gemv", "vocab", "sample"])
    heads, kv = rng.choice([(40, 8), (32, 2)])
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16"])
    if kind == "norm":
        return {"kind": kind, "tokens": _log(rng, 1, 4096), "dim": rng.choice([5120, 6656]), "dtype": dtype}
    if kind == "swiglu":
        return {"kind": kind, "tokens": _log(rng, 1, 4096), "ffn": rng.choice([25600, 19968]), "dtype": dtype}
    if kind == "qk":
        return {"kind": kind, "tokens": _log(rng, 1, 4096), "heads": heads, "kv": kv, "pos0": rng.randrange(0, 4096)}
    if kind == "softmax":
        k = _log(rng, 64, 16384)
        q = _log(rng, 1, max(1, min(k, 2048, 160_000_000 // (heads * k))))
        return {"kind": kind, "heads": heads, "q": q, "k": k, "pos0": k - q,
                "window": rng.choice([0, 0, 0, 1024]), "cap": rng.choice([0.0, 0.0, 30.0])}
    if kind == "prefill":
        tokens = _log(rng, 2, 4096)
        # no more pairs than the largest listed call has
        most = min(32768, max(0, (40 * 4096 * 2048 // heads) // tokens - tokens))
        return {"kind": kind, "tokens": tokens, "heads": heads, "kv": kv, "pos0": rng.randrange(0, most + 1),
                "window": rng.choice([0, 0, 0, 1024])}
    if kind == "decode":
        return {"kind": kind, "heads": heads, "kv": kv, "keys": _log(rng, 64, 131072)}
    if kind == "gemv":
        rows, n = rng.choice([(25600, 5120), (5120, 25600), (19968, 6656), (6656, 19968), (5120, 5120), (1024, 5120)])
        return {"kind": kind, "rows": rows, "in": n, "batch": rng.randrange(1, 9)}
    if kind == "vocab":
        return {"kind": kind, "rows": _log(rng, 1, 64), "V": rng.choice([201088, 202048]),
                "K": rng.choice([20, 40, 64]), "top_p": round(rng.uniform(0.8, 0.99), 3)}
    return {"kind": kind, "rows": _log(rng, 1, 64), "V": rng.choice([201088, 202048]),
            "top_p": round(rng.uniform(0.8, 0.95), 3), "min_p": rng.choice([0.0, 0.0, 0.01])}


# ------------------------------------------------------------------- inputs
def _slots(c):
    """Ring size of an attention call: its keys, rounded up as a cache is allocated."""
    n = c["pos0"] + c["tokens"] if c["kind"] != "decode" else c["keys"]
    return (n + 255) // 256 * 256


def _inputs(c, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1_000_003 * (seed % 1_000_000_007) + 17)

    def randn(shape, mean=0.0, std=1.0, dtype=torch.bfloat16):
        return (torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * std + mean).to(dtype)

    k, s = c["kind"], {}
    if k == "norm":
        dt = DTYPES[c["dtype"]]
        s["h"], s["x"] = (randn((c["tokens"], c["dim"]), dtype=dt) for _ in range(2))
        s["w"] = randn((c["dim"],), 1.0, 0.05, dt)
    elif k == "swiglu":
        s["gate"], s["up"] = (randn((c["tokens"], c["ffn"]), dtype=DTYPES[c["dtype"]]) for _ in range(2))
    elif k == "qk":
        s["q"] = randn((c["tokens"], c["heads"], HD))
        s["k"], s["v"] = (randn((c["tokens"], c["kv"], HD)) for _ in range(2))
    elif k == "softmax":
        # softcapped scores run wide enough that the cap bends them
        s["x"] = randn((c["heads"], c["q"], c["k"]), 0.0, 60.0 if c["cap"] else 3.0, torch.float32)
    elif k == "prefill":
        s["q"] = randn((c["tokens"], c["heads"], HD))
        s["k"], s["v"] = (randn((_slots(c), c["kv"], HD)) for _ in range(2))
    elif k == "decode":
        s["q"] = randn((c["heads"], HD))
        s["k"], s["v"] = (randn((_slots(c), c["kv"], HD)) for _ in range(2))
    elif k == "gemv":
        s["qs"] = torch.randint(-127, 128, (c["rows"], c["in"]), generator=g, device=DEV, dtype=torch.int8)
        s["d"] = (torch.rand((c["rows"], c["in"] // 32), generator=g, device=DEV) * (2e-2 - 1e-3) + 1e-3).half()
        s["x"] = randn((c["batch"], c["in"]))
    else:
        s["logits"] = randn((c["rows"], c["V"]), 0.0, 4.0, torch.float32)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"], s["P"] = case, prims()
    k = case["kind"]

    def empty(shape, dtype):
        return torch.empty(shape, dtype=dtype, device=DEV)

    if k == "norm":
        s["y"] = torch.empty_like(s["h"])
    elif k == "swiglu":
        s["out"] = torch.empty_like(s["gate"])
    elif k == "qk":
        s["cos"], s["sin"] = s["P"].build_rope_table(THETA, HD, case["pos0"] + case["tokens"], torch.bfloat16)
        s["kc"], s["vc"] = (torch.zeros((_slots(case), case["kv"], HD), dtype=torch.bfloat16, device=DEV)
                            for _ in range(2))
    elif k == "softmax":
        s["y"] = empty(s["x"].shape, torch.bfloat16)
    elif k in ("prefill", "decode"):
        s["out"] = empty(s["q"].shape, torch.float32)
    elif k == "gemv":
        s["y"] = empty((case["batch"], case["rows"]), torch.float32)
    elif k == "vocab":
        # slots past a row's count keep what they held
        s["ids"] = torch.zeros((case["rows"], case["K"]), dtype=torch.int64, device=DEV)
        s["probs"] = torch.zeros((case["rows"], case["K"]), dtype=torch.float32, device=DEV)
    else:
        s["slot"] = torch.arange(SAMPLE_MAX, device=DEV)
    return s


SAMPLE_MAX = 4096  # candidates a sorted row can hold (mg_sample_rows)


# --------------------------------------------------------------------- pass
def run(s):
    c, P = s["case"], s["P"]
    k = c["kind"]
    if k == "norm":
        P.residual_rmsnorm(M.PLAIN, s["h"], s["x"], s["w"], EPS, s["y"])
        return s["h"], s["y"]
    if k == "swiglu":
        P.swiglu(s["gate"], s["up"], s["out"])
        return s["out"]
    if k == "qk":
        P.qk_norm_rope(s["q"], s["k"], EPS, QK_SCALE, s["cos"], s["sin"], None, c["pos0"], s["v"], s["kc"], s["vc"])
        return s["q"], s["k"], s["kc"], s["vc"]
    if k == "softmax":
        P.softmax_rows(s["x"], s["y"], SCALE, M.MASK_WINDOW if c["window"] else M.MASK_CAUSAL, c["window"], c["pos0"],
                       c["cap"])
        return s["y"]
    if k == "prefill":
        return P.attn_prefill(s["q"], s["k"], s["v"], c["pos0"], SCALE, c["window"], s["out"])
    if k == "decode":
        return P.attn_decode(s["q"], s["k"], s["v"], c["keys"] - 1, SCALE, 0, s["out"])
    if k == "gemv":
        P.gemv_q8_0(s["qs"], s["d"], s["x"], s["y"])
        return s["y"]
    if k == "vocab":
        lse, amax, ti, tv = P.vocab_reduce_tail(s["logits"], 1.0, 30.0, c["K"])
        ids, probs, n = P.sample_dist(ti, tv, amax, 0.7, c["top_p"], 0.0, s["ids"], s["probs"])
        return lse, amax, ti, tv, ids, probs, n
    ids, probs, n = P.sample_rows(s["logits"], 0, 1.0, c["top_p"], c["min_p"])
    # the slots past a row's count are not written: a draw masks them
    live = s["slot"] < n[:, None]
    return torch.where(live, ids[:, :SAMPLE_MAX], -1), torch.where(live, probs[:, :SAMPLE_MAX], 0.0), n


# ------------------------------------------------------------------ measure
def _pairs(c):
    """Visible (query, key) pairs of one head: causal, or the window's keys."""
    t, p, w = c.get("tokens", c.get("q")), c["pos0"], c["window"]
    if not w:
        return t * p + t * (t + 1) // 2
    return sum(min(w, p + i + 1) for i in range(t))


def work(c):
    k = c["kind"]
    if k == "norm":
        n = c["tokens"] * c["dim"]
        return {"bytes": 4 * 2 * n + 2 * c["dim"], "flops": 6 * n}
    if k == "swiglu":
        n = c["tokens"] * c["ffn"]
        return {"bytes": 3 * 2 * n, "flops": 6 * n}
    if k == "qk":
        q, kk, t = c["tokens"] * c["heads"] * HD, c["tokens"] * c["kv"] * HD, c["tokens"] * HD // 2
        return {"bytes": 2 * 2 * (q + kk) + 2 * kk + 2 * 2 * kk + 2 * 2 * t, "flops": 10 * (q + kk)}
    if k == "softmax":
        seen = c["heads"] * _pairs(c)
        return {"bytes": 4 * seen + 2 * c["heads"] * c["q"] * c["k"], "flops": 5 * seen}
    if k == "prefill":
        q = c["tokens"] * c["heads"] * HD
        keys = min(c["pos0"] + c["tokens"], c["window"] + c["tokens"] - 1 if c["window"] else 1 << 60)
        return {"bytes": 2 * q + 4 * q + 2 * 2 * keys * c["kv"] * HD, "flops": 4 * HD * c["heads"] * _pairs(c)}
    if k == "decode":
        return {"bytes": 2 * 2 * c["keys"] * c["kv"] * HD + 6 * c["heads"] * HD, "flops": 4 * HD * c["heads"] * c["keys"]}
    if k == "gemv":
        n = c["rows"] * c["in"]
        return {"bytes": n + 2 * (n // 32) + 2 * c["batch"] * c["in"] + 4 * c["batch"] * c["rows"],
                "flops": 2 * n * c["batch"]}
    n = c["rows"] * c["V"]
    if k == "vocab":
        return {"bytes": 4 * n + c["rows"] * (24 + 2 * 12 * c["K"]), "flops": 8 * n}
    return {"bytes": 4 * n + c["rows"] * 8, "flops": 5 * n}


def tolerance(c):
    k = c["kind"]
    # the gating and the QK chain are defined to the bit: one rounding a step, in a given order
    if k in ("swiglu", "qk"):
        return "exact"
    # f64 sums, one rounding to 16 bits: a value at a rounding boundary may fall to either side
    if k == "norm":
        return {"rel": 4e-3, "max": 1e-2}
    # bf16 probabilities: one ulp
    if k == "softmax":
        return {"rel": 7e-3, "max": 1e-2}
    # bf16 weights in the second product (2^-9 rms each, independent), f32 sums
    if k == "prefill":
        return {"rel": 7e-3, "max": 5e-2}
    # weights to 2^-16, f32 sums
    if k == "decode":
        return {"rel": 4e-5, "max": 4e-4}
    # f32 sums of thousands of products
    if k == "gemv":
        return {"rel": 4e-6, "max": 4e-5}
    # f32 exponentials, f64 sums; ids are exact selections, a cut may fall one candidate apart
    return {"rel": 4e-6, "max": 4e-5, "differ": 2e-3}


# ------------------------------------------------------------- 64-bit result
def _norm64(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _attn64(q, k, v, pos0, window):
    """f64 attention of q [T, Hq, D] over keys [n, Hk, D], head by head."""
    T, hq, _ = q.shape
    n, hk, _ = k.shape
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    qpos = pos0 + torch.arange(T, device=q.device)[:, None]
    key = torch.arange(n, device=q.device)[None, :]
    hidden = key > qpos
    if window:
        hidden |= key <= qpos - window
    for h in range(hq):
        gk, gv = (t[:, h // (hq // hk), :].double().contiguous() for t in (k, v))
        sc = (q[:, h, :].double() @ gk.t().contiguous()) * SCALE
        out[:, h, :] = torch.softmax(sc.masked_fill_(hidden, -math.inf), -1) @ gv
    return out


def _rope64(x, cos, sin):
    lo, hi = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat((lo * cos - hi * sin, hi * cos + lo * sin), -1)


def _dist64(val, idx, temperature, top_p, min_p, width):
    """The kept candidates of rows sorted by value: (ids, probs, n), `width` slots a row."""
    p = torch.softmax(val, -1)
    n = (p.cumsum(-1) < top_p).sum(-1) + 1
    n = torch.minimum(n, (p >= min_p * p[:, :1]).sum(-1))
    live = torch.arange(width, device=val.device)[None, :] < n[:, None]
    f = torch.softmax((val[:, :width] / temperature).masked_fill(~live, -math.inf), -1)
    return live, idx[:, :width], f, n


def exact(case, seed):
    c, s = case, _inputs(case, seed)
    k = c["kind"]
    if k == "norm":
        h = s["h"].double() + s["x"].double()
        return h, _norm64(h.to(s["h"].dtype).double()) * s["w"].double()
    if k == "swiglu":
        g = s["gate"].double()
        return g * torch.sigmoid(g) * s["up"].double()
    if k == "qk":
        inv = THETA ** (-torch.arange(0, HD, 2, dtype=torch.float64, device=DEV) / HD)
        pos = c["pos0"] + torch.arange(c["tokens"], dtype=torch.float64, device=DEV)
        ang = (pos[:, None] * inv)[:, None, :]
        q = _rope64(_norm64(s["q"].double()) * QK_SCALE, ang.cos(), ang.sin())
        kk = _rope64(_norm64(s["k"].double()), ang.cos(), ang.sin())
        kc, vc = (torch.zeros((_slots(c), c["kv"], HD), dtype=torch.float64, device=DEV) for _ in range(2))
        kc[c["pos0"]:c["pos0"] + c["tokens"]] = kk
        vc[c["pos0"]:c["pos0"] + c["tokens"]] = s["v"].double()
        return q, kk, kc, vc
    if k == "softmax":
        out = torch.empty(s["x"].shape, dtype=torch.float64, device=DEV)
        qpos = c["pos0"] + torch.arange(c["q"], device=DEV)[:, None]
        key = torch.arange(c["k"], device=DEV)[None, :]
        hidden = key > qpos
        if c["window"]:
            hidden |= key <= qpos - c["window"]
        for h in range(c["heads"]):
            x = s["x"][h].double() * SCALE
            if c["cap"]:
                x = torch.tanh(x / c["cap"]) * c["cap"]
            out[h] = torch.softmax(x.masked_fill_(hidden, -math.inf), -1)
        return out
    if k == "prefill":
        n = c["pos0"] + c["tokens"]
        return _attn64(s["q"], s["k"][:n], s["v"][:n], c["pos0"], c["window"])
    if k == "decode":
        n = c["keys"]
        return _attn64(s["q"][None], s["k"][:n], s["v"][:n], n - 1, 0)[0]
    if k == "gemv":
        # the weights are defined as bf16(q * d)
        w = (s["qs"].float() * s["d"].float().repeat_interleave(32, 1)).bfloat16()
        y = torch.empty((c["batch"], c["rows"]), dtype=torch.float64, device=DEV)
        for i in range(0, c["rows"], 2048):
            y[:, i:i + 2048] = s["x"].double() @ w[i:i + 2048].double().t().contiguous()
        return y
    if k == "vocab":
        # the tail is defined step by step with an f32 rounding each: ties among its values count
        t = torch.tanh((s["logits"] / 30.0).double()).float()
        z = (30.0 * t).double()
        val, idx = torch.sort(z, dim=-1, descending=True, stable=True)
        live, ids, f, n = _dist64(val[:, :c["K"]], idx[:, :c["K"]], 0.7, c["top_p"], 0.0, c["K"])
        return (torch.logsumexp(z, -1), idx[:, 0].contiguous(), idx[:, :c["K"]], val[:, :c["K"]],
                torch.where(live, ids, 0), torch.where(live, f, 0.0), n)
    val, idx = torch.sort(s["logits"].double(), dim=-1, descending=True, stable=True)
    live, ids, f, n = _dist64(val, idx, 1.0, c["top_p"], c["min_p"], SAMPLE_MAX)
    return torch.where(live, ids, -1), torch.where(live, f, 0.0), n
