"""Performance cases of the kernel layer: what a program that serves a Dory-shaped model has it do.

The shapes are the two model configurations of xtier-go_amd/workloads.py (the 4B-shaped one: hidden 3072, 32 / 8 heads
of 128, FFN 8192; the real one: hidden 2560, 16 / 4 heads of 256, FFN 7168), at the row counts of its calls: 1 row (a
decode step), 2-8 rows (a speculative verify step), the ragged tail of a prompt, a full 512-row prompt chunk, and the
longer calls the device matmul takes. Weights are E2M1 codes with E4M3 scales drawn as that file draws them; caches hold
unit keys, and queries are scaled so that a row's scores spread over several units.

A case is a dict of plain values; prepare() makes what a program holds before the call (weights prepared on the device,
caches filled, device buffers), run() is one pass through the public entry points, exact() the same outputs in 64 bits
from plain torch.
"""
import importlib
import math
import os
import sys

import numpy as np
import torch

E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)

# The projection groups of the two configurations that one call computes: (output rows of each weight, inputs).
PROJ = {
    "qkvg-3072": "4096+1024+1024+4096x3072", "gateup-3072": "8192+8192x3072", "o-3072": "3072x4096",
    "down-3072": "3072x8192", "qkvg-2560": "4096+1024+1024+4096x2560", "gateup-2560": "7168+7168x2560",
    "o-2560": "2560x4096", "down-2560": "2560x7168",
}

# Models of a quarter of the depth of the two configurations (the widths, heads, window, loops, KV modes and heads are
# theirs): a decode step's cost is per sublayer, and 16 sublayers hold two global attention layers.
MODELS = {
    "4b": dict(hidden=3072, ffn=8192, heads=32, kv_heads=8, head_dim=128, vocab=131072, n_in=4, n_rec=8, n_out=4,
               loops=1, window=1024, ring_slots=1088, theta_sliding=1e6, theta_full=1e6),
    "real": dict(hidden=2560, ffn=7168, heads=16, kv_heads=4, head_dim=256, vocab=131072, n_in=4, n_rec=8, n_out=4,
                 loops=2, window=1024, ring_slots=1040, theta_sliding=1e4, theta_full=1e7, kv_dtype=1, kv_mode=1,
                 bf16_head=True),
}
MLP, SLIDING, FULL = 0, 1, 2


def listed():
    return [
        # the projections of one decoded token: the smallest call, one launch over 18 MB of weights
        {"name": "qkvg-1row", "kind": "proj", "shape": PROJ["qkvg-3072"], "m": 1, "x": "bf16"},
        # a speculative verify step's widest projection, on FP32 rows
        {"name": "gateup-8rows", "kind": "proj", "shape": PROJ["gateup-2560"], "m": 8, "x": "f32"},
        # the ragged tail of a prompt (or a short prompt)
        {"name": "o-37rows", "kind": "proj", "shape": PROJ["o-3072"], "m": 37, "x": "f32"},
        # a full prompt chunk's widest projection
        {"name": "gateup-512rows", "kind": "proj", "shape": PROJ["gateup-3072"], "m": 512, "x": "f32"},
        # a long device call, not a multiple of anything
        {"name": "down-1500rows", "kind": "proj", "shape": PROJ["down-2560"], "m": 1500, "x": "bf16"},
        # the BF16 checkpoint's LM head over a few rows of a verify step
        {"name": "head-bf16-4rows", "kind": "head", "vocab": 131072, "k": 2560, "m": 4, "x": "f32"},
        # one token's attention over a long BF16 cache (a global layer of the 4B-shaped model)
        {"name": "attn-1row-32k", "kind": "attn", "n_q": 1, "ctx": 32768, "heads": 32, "kv_heads": 8, "d": 128,
         "ring": 0, "window": 0, "fp8": False},
        # a verify step's attention over a full FP8 ring (a sliding layer of the real model)
        {"name": "attn-8rows-ring-fp8", "kind": "attn", "n_q": 8, "ctx": 5000, "heads": 16, "kv_heads": 4, "d": 256,
         "ring": 1040, "window": 1024, "fp8": True},
        # a prompt chunk's attention in the middle of a prompt
        {"name": "attn-512rows-3k", "kind": "attn", "n_q": 512, "ctx": 3000, "heads": 32, "kv_heads": 8, "d": 128,
         "ring": 0, "window": 0, "fp8": False},
        # one sampled token at the usual serving settings
        {"name": "sample-top-p", "kind": "sample", "rows": 1, "n": 131072, "t": 0.8, "top_p": 0.95, "top_k": 0,
         "min_p": 0.0},
        # a decode step of a model: 4K context, BF16 caches, NVFP4 head
        {"name": "step-4b-4k", "kind": "model", "model": "4b", "m": 1, "ctx": 4096},
        # a prompt of a model: a full chunk and a ragged one, two loops, FP8 caches, the last row's logits
        {"name": "prompt-real-700", "kind": "model", "model": "real", "m": 700, "ctx": 0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["proj", "proj", "proj", "proj", "attn", "attn", "attn", "head", "sample", "model", "model"])
    if kind == "proj":
        if rng.random() < 0.75:
            shape = PROJ[rng.choice(sorted(PROJ))]
        else:   # any widths: one to three weights of an odd number of rows, inputs in whole scale groups
            shape = "+".join(str(_log(rng, 500, 8000)) for _ in range(rng.randint(1, 3)))
            shape += "x%d" % (16 * _log(rng, 16, 512))
        m = _log(rng, 1, 8) if rng.random() < 0.4 else _log(rng, 9, 2048)
        return {"kind": "proj", "shape": shape, "m": m, "x": rng.choice(["f32", "bf16"])}
    if kind == "head":
        return {"kind": "head", "vocab": rng.choice([131072, 50257, 32000]), "k": rng.choice([2560, 3072]),
                "m": rng.randint(1, 8), "x": rng.choice(["f32", "bf16"])}
    if kind == "attn":
        heads, kv, d = rng.choice([(32, 8, 128), (16, 4, 256), (32, 8, 128), (16, 4, 256), (16, 8, 64)])
        n_q = rng.choice([1, _log(rng, 2, 8), _log(rng, 9, 512), _log(rng, 9, 512)])
        ring = rng.random() < 0.5
        return {"kind": "attn", "n_q": n_q, "ctx": _log(rng, 500, 32768 if n_q <= 8 else 8192), "heads": heads,
                "kv_heads": kv, "d": d, "ring": (1040 if d == 256 else 1088) if ring else 0,
                "window": 1024 if ring else 0, "fp8": rng.random() < 0.5}
    if kind == "sample":
        return {"kind": "sample", "rows": rng.randint(1, 8), "n": rng.choice([131072, 50257, 32000]),
                "t": rng.choice([0.0, 0.6, 0.8, 1.0]), "top_p": rng.choice([1.0, 0.95, 0.8]),
                "top_k": rng.choice([0, 0, 20, 64, 200]), "min_p": rng.choice([0.0, 0.0, 0.05])}
    model = rng.choice(["4b", "real"])
    m = rng.choice([1, rng.randint(2, 8), _log(rng, 9, 640)])
    return {"kind": "model", "model": model, "m": m, "ctx": _log(rng, 500, 16384) if m <= 8 else 0}


# ------------------------------------------------------------------------------------------------------- inputs


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _nvfp4(g, n, k):
    """(codes [n][k/2], scales [n][k/16]) on the GPU: uniform codes, scales |N(0,1)| * 0.05 rounded to E4M3."""
    codes = torch.randint(0, 256, (n, k // 2), generator=g, device="cuda", dtype=torch.uint8)
    s = torch.randn((n, k // 16), generator=g, device="cuda").abs() * 0.05
    return codes, s.to(torch.float8_e4m3fn).view(torch.uint8)


def _bf16_weight(g, n, k):
    return torch.randn((n, k), generator=g, device="cuda", dtype=torch.bfloat16)


def _unit(g, shape):
    x = torch.randn(shape, generator=g, device="cuda")
    return x / x.norm(dim=-1, keepdim=True)


def _rows(g, m, k, x):
    r = _unit(g, (m, k))
    return r.bfloat16() if x == "bf16" else r


def _shape(s):
    n, k = s.split("x")
    return [int(v) for v in n.split("+")], int(k)


def _proj_inputs(case, seed):
    g = _gen(seed)
    ns, k = _shape(case["shape"])
    return [_nvfp4(g, n, k) for n in ns], _rows(g, case["m"], k, case["x"])


def _attn_inputs(case, seed):
    """Cached K, V [ctx][kv][d], and the call's q, k, v."""
    g = _gen(seed)
    n, ctx, d = case["n_q"], case["ctx"], case["d"]
    kc = _unit(g, (ctx, case["kv_heads"], d))
    vc = torch.randn((ctx, case["kv_heads"], d), generator=g, device="cuda")
    q = _unit(g, (n, case["heads"], d)) * d * (0.5 + torch.rand((1, case["heads"], d), generator=g, device="cuda"))
    return kc, vc, q, _unit(g, (n, case["kv_heads"], d)), torch.randn((n, case["kv_heads"], d), generator=g,
                                                                     device="cuda")


def _sample_inputs(case, seed):
    g = _gen(seed)
    logits = torch.randn((case["rows"], case["n"]), generator=g, device="cuda") * 3.0
    u = torch.rand((case["rows"],), generator=g, device="cuda", dtype=torch.float64).cpu().numpy()
    return logits, u


def _kinds(c):
    """Attention and MLP alternate, attention first; every fourth attention sublayer is global."""
    return [MLP if l % 2 else FULL if (l // 2) % 4 == 3 else SLIDING for l in range(c["n_in"] + c["n_rec"] + c["n_out"])]


def _model_inputs(case, seed):
    """(config, layers, head, logit scale, rows, [(K, V) of each attention sublayer's cached context])."""
    c = dict(MODELS[case["model"]])
    c["context"] = case["ctx"] + case["m"] + 64
    g = _gen(seed)
    H, F = c["hidden"], c["ffn"]
    Q, KV = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]

    def uniform(lo, hi, n):
        return lo + (hi - lo) * torch.rand(n, generator=g, device="cuda")

    layers, cached = [], []
    for kind in _kinds(c):
        L = {"kind": kind, "lr": uniform(0.02, 0.1, H)}
        if kind == MLP:
            L.update(gate=_nvfp4(g, F, H), up=_nvfp4(g, F, H), down=_nvfp4(g, H, F), sg=uniform(5, 15, F),
                     su=uniform(5, 15, F))
        else:
            L.update(q=_nvfp4(g, Q, H), k=_nvfp4(g, KV, H), v=_nvfp4(g, KV, H), g=_nvfp4(g, Q, H), o=_nvfp4(g, H, Q),
                     qscale=uniform(0.5, 1.5, Q) * c["head_dim"], gscale=uniform(0.5, 1.5, Q))
            # a ring of a long context holds its last positions only
            n = case["ctx"] if kind == FULL else min(case["ctx"], c["ring_slots"])
            cached.append((_unit(g, (n, c["kv_heads"], c["head_dim"])),
                           torch.randn((n, c["kv_heads"], c["head_dim"]), generator=g, device="cuda")))
        layers.append(L)
    head = _bf16_weight(g, c["vocab"], H) if c.get("bf16_head") else _nvfp4(g, c["vocab"], H)
    x = _unit(g, (case["m"], H))
    return c, layers, head, uniform(0.5, 1.5, c["vocab"]), x, cached


# ---------------------------------------------------------------------------------------------- the framework's side

_backend = []


def _package():
    """The package under the name its own modules use, from the tree that is the working folder."""
    if "xtier_go_amd" not in sys.modules:
        if os.getcwd() not in sys.path:
            sys.path.insert(0, os.getcwd())
        sys.modules["xtier_go_amd"] = importlib.import_module("xtier-go_amd")
    return sys.modules["xtier_go_amd"]


def _hip():
    """The one backend (device, stream and prepared weights) that a program keeps open."""
    if not _backend:
        _backend.append(_package().HipBackend(0))
    return _backend[0]


class _State:
    """What one program holds; its device copies go with it."""

    def __init__(self, case):
        self.case, self.b = case, _hip()
        self.weights, self.heads, self.cache, self.session = [], [], None, None

    def weight(self, w):
        pkg = _package()
        self.weights.append(pkg.Weight(w[0].cpu().numpy(), w[1].cpu().numpy(), 1.0))
        self.b.prepare(self.weights[-1])
        return self.weights[-1]

    def __del__(self):
        if self.session is not None:
            self.session.destroy()
        if self.cache is not None:
            self.cache.destroy()
        for w in self.weights:
            self.b.release_weight(w)
        for w in self.heads:
            self.b.release_bf16(w)


class _ModelWeights:
    """The host side of a model that a Dory session is made from (the fields of workloads.DoryWeights)."""

    def __init__(self, c, layers, head, logit_scale):
        def host(v):
            if isinstance(v, tuple):
                return v[0].cpu().numpy(), v[1].cpu().numpy(), 1.0
            return v.cpu().numpy() if isinstance(v, torch.Tensor) else v

        self.cfg, self.kinds = c, _kinds(c)
        self.layers = [{name: host(v) for name, v in L.items()} for L in layers]
        self.logit_scale = logit_scale.cpu().numpy()
        self.head, self.head_bf16 = None, None
        if c.get("bf16_head"):
            self.head_bf16 = head.view(torch.int16).cpu().numpy().view(np.uint16)
        else:
            self.head = host(head)


def prepare(case, seed):
    s = _State(case)
    kind = case["kind"]
    if kind == "proj":
        ws, s.x = _proj_inputs(case, seed)
        s.ws = [s.weight(w) for w in ws]
        s.y = torch.zeros(case["m"] * sum(w.n_out for w in s.ws), device="cuda")
        s.dtype = _package().X_BF16 if case["x"] == "bf16" else _package().X_F32
    elif kind == "head":
        g = _gen(seed)
        w = _bf16_weight(g, case["vocab"], case["k"])
        s.x = _rows(g, case["m"], case["k"], case["x"])
        s.w = w.view(torch.int16).cpu().numpy().view(np.uint16)
        s.b.prepare_bf16(s.w)
        s.heads.append(s.w)
        s.y = torch.zeros((case["m"], case["vocab"]), device="cuda")
        s.dtype = _package().X_BF16 if case["x"] == "bf16" else _package().X_F32
    elif kind == "attn":
        kc, vc, s.q, s.k, s.v = _attn_inputs(case, seed)
        torch.cuda.synchronize()
        s.cache = s.b.kv_cache(case["kv_heads"], case["d"], case["ctx"] + case["n_q"], case["ring"],
                               _package().KV_FP8 if case["fp8"] else _package().KV_BF16)
        s.cache.store(0, case["ctx"], kc, vc)
        s.b.finish()
        s.out = torch.zeros_like(s.q)
    elif kind == "sample":
        s.logits, s.u = _sample_inputs(case, seed)
        s.out = torch.zeros(case["rows"], device="cuda", dtype=torch.int32)
    else:
        c, layers, head, logit_scale, s.x, cached = _model_inputs(case, seed)
        s.session = s.b.dory(_ModelWeights(c, layers, head, logit_scale))
        torch.cuda.synchronize()
        for a, (k, v) in enumerate(cached):
            for inst in range(c["loops"] if c.get("kv_mode", 0) == 0 and _recurrent(c, 2 * a) else 1):
                if k.shape[0]:
                    s.session.cache(a, inst).store(case["ctx"] - k.shape[0], k.shape[0], k, v)
        s.b.finish()
        s.logits = torch.zeros((case["m"] if case["m"] <= 8 else 1, c["vocab"]), device="cuda")
    torch.cuda.synchronize()
    return s


def run(s):
    case, kind = s.case, s.case["kind"]
    if kind == "proj":
        s.b.matmul_dev(s.ws, s.x, s.dtype, case["m"], s.y)
        return s.y
    if kind == "head":
        s.b.matmul_bf16_dev(s.w, s.x, s.dtype, case["m"], s.y)
        return s.y
    if kind == "attn":
        s.b.attention(s.cache, s.q, s.k, s.v, s.out, case["n_q"], case["ctx"], case["heads"], case["window"])
        return s.out
    if kind == "sample":
        s.b.sample(s.logits, case["rows"], case["n"], s.u, s.out, case["t"], case["top_p"], case["top_k"],
                   case["min_p"])
        return s.out
    if case["m"] <= 8:   # a decode or verify step: logits of every row
        s.session.forward(s.x, case["m"], case["ctx"], s.logits)
    else:                # a prompt: the last row's logits
        s.session.prefill(s.x, case["m"], case["ctx"], _package().LOGITS_LAST, s.logits)
    return s.logits


# ---------------------------------------------------------------------------------------------------- what is needed


def _weight_bytes(n, k):
    return n * k // 2 + n * k // 16


def _visible(case_ctx, n_q, window):
    """Query-key pairs of a causal call of n_q rows after case_ctx positions."""
    return sum(min(case_ctx + i + 1, window) if window else case_ctx + i + 1 for i in range(n_q))


def _attn_work(n_q, ctx, heads, kv, d, window, fp8):
    seen = min(ctx, window + n_q - 1) if window else ctx
    row = kv * (d + 4 if fp8 else 2 * d) * 2
    return {"bytes": seen * row + 4 * n_q * d * (2 * heads + 2 * kv),
            "flops": 4 * d * heads * _visible(ctx, n_q, window)}


def work(case):
    kind = case["kind"]
    if kind == "proj":
        ns, k = _shape(case["shape"])
        m = case["m"]
        return {"bytes": sum(_weight_bytes(n, k) for n in ns) + m * k * (2 if case["x"] == "bf16" else 4) + 4 * m * sum(ns),
                "flops": 2 * m * k * sum(ns)}
    if kind == "head":
        n, k, m = case["vocab"], case["k"], case["m"]
        return {"bytes": 2 * n * k + m * k * (2 if case["x"] == "bf16" else 4) + 4 * m * n, "flops": 2 * m * n * k}
    if kind == "attn":
        return _attn_work(case["n_q"], case["ctx"], case["heads"], case["kv_heads"], case["d"], case["window"],
                          case["fp8"])
    if kind == "sample":
        return {"bytes": 4 * case["rows"] * case["n"], "flops": 0}
    c, m = MODELS[case["model"]], case["m"]
    H, F, d = c["hidden"], c["ffn"], c["head_dim"]
    Q, KV = c["heads"] * d, c["kv_heads"] * d
    fp8 = bool(c.get("kv_dtype", 0))
    out = m if m <= 8 else 1
    total = {"bytes": (2 * c["vocab"] * H if c.get("bf16_head") else _weight_bytes(c["vocab"], H)) + 4 * out * c["vocab"],
             "flops": 2 * out * H * c["vocab"]}
    for l, kind in enumerate(_kinds(c)):
        times = c["loops"] if _recurrent(c, l) else 1
        if kind == MLP:
            w = [(2 * F, H), (H, F)]
        else:
            w = [(2 * Q + 2 * KV, H), (H, Q)]
            a = _attn_work(m, case["ctx"], c["heads"], c["kv_heads"], d, c["window"] if kind == SLIDING else 0, fp8)
            # q, k, v and the output stay on the chip: the cached rows and the new ones' stores count
            total["bytes"] += times * (a["bytes"] - 4 * m * d * (2 * c["heads"] + 2 * c["kv_heads"]))
            total["bytes"] += m * c["kv_heads"] * (d + 4 if fp8 else 2 * d) * 2
            total["flops"] += times * a["flops"]
        total["bytes"] += times * sum(_weight_bytes(n, k) for n, k in w)
        total["flops"] += times * sum(2 * m * n * k for n, k in w)
    return total


def _recurrent(c, l):
    return c["n_in"] <= l < c["n_in"] + c["n_rec"]


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":   # token numbers
        return "exact"
    # about four times the 2-norm distance to the 64-bit result that the path shows, over the sizes of draw()
    if kind == "model":   # FP32 rows through 16 sublayers (24 with the second loop); a cached key may round to its neighbour
        return {"rel": 1.2e-4, "max": 2e-3} if case["m"] > 8 else {"rel": 3e-5, "max": 5e-4}
    if kind == "attn":    # scores of 24 bits, softmax weights of 16
        return {"rel": 1e-5, "max": 2e-4}
    if kind == "proj" and case["x"] == "bf16" and case["m"] <= 2:   # block-scaled products, sums per scale group
        return {"rel": 1.5e-5, "max": 2e-4}
    return {"rel": 1.5e-6, "max": 3e-5}   # FP32 sums of exact products, activations in about 22 bits


# ------------------------------------------------------------------------------------------------------ in 64 bits


def _dense(w):
    """An NVFP4 weight's values [n][k] in 64 bits."""
    codes, scales = w
    t = torch.tensor(E2M1 + tuple(-v for v in E2M1), device=codes.device, dtype=torch.float64)
    v = torch.stack((t[(codes & 15).long()], t[(codes >> 4).long()]), dim=-1).reshape(codes.shape[0], -1)
    return v * scales.view(torch.float8_e4m3fn).double().repeat_interleave(16, dim=1)


def _times(x, w):
    """x [m][k] times an NVFP4 or BF16 weight, in blocks of its rows."""
    out, step = [], 16384
    n = w[0].shape[0] if isinstance(w, tuple) else w.shape[0]
    for r in range(0, n, step):
        part = _dense((w[0][r:r + step], w[1][r:r + step])) if isinstance(w, tuple) else w[r:r + step].double()
        out.append(x @ part.T)
    return torch.cat(out, dim=1)


def _stored(x, fp8):
    """A row as the cache holds it: BF16, or E4M3 codes with the scale amax / 448 per (position, head)."""
    x = x.float()
    if not fp8:
        return x.bfloat16().double()
    amax = x.abs().amax(dim=-1, keepdim=True)
    s = torch.where(amax > 0, amax / 448.0, torch.ones_like(amax))
    return ((x * (1.0 / s)).clamp(-448, 448).to(torch.float8_e4m3fn).double()) * s.double()


def _attend(q, k, v, kc, vc, pos0, p0, window):
    """Causal attention of q [m][heads][d] at pos0 .. over cached rows (positions p0 ..) and the call's own k, v."""
    m, heads, d = q.shape
    group = heads // k.shape[1]
    at = torch.cat((torch.arange(p0, p0 + kc.shape[0], device=q.device), torch.arange(pos0, pos0 + m, device=q.device)))
    mine = torch.arange(pos0, pos0 + m, device=q.device)[:, None]
    hide = at[None, :] > mine
    if window:
        hide = hide | (mine - at[None, :] >= window)
    out = torch.empty_like(q)
    for h in range(k.shape[1]):
        kk, vv = torch.cat((kc[:, h], k[:, h])), torch.cat((vc[:, h], v[:, h]))
        for j in range(h * group, (h + 1) * group):
            p = ((q[:, j] @ kk.T) / math.sqrt(d)).masked_fill(hide, -math.inf).softmax(dim=-1)
            out[:, j] = p @ vv
    return out


def _justnorm(x):
    return x / (x.square().sum(dim=-1, keepdim=True) + 1e-6).sqrt()


def _rope(x, pos0, theta):
    """NeoX RoPE of [m][heads][d]; the angles are 32-bit products, as the model defines them."""
    m, _, d = x.shape
    freq = torch.tensor([np.float32(1) / np.power(np.float32(theta), np.float32(2 * i) / np.float32(d), dtype=np.float32)
                         for i in range(d // 2)], dtype=torch.float32, device=x.device)
    a = (torch.arange(pos0, pos0 + m, device=x.device).float()[:, None] * freq[None, :]).double()[:, None, :]
    lo, hi = x[..., :d // 2], x[..., d // 2:]
    return torch.cat((lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin()), dim=-1)


def _model_exact(case, seed):
    c, layers, head, logit_scale, rows, cached = _model_inputs(case, seed)
    heads, kv, d, fp8 = c["heads"], c["kv_heads"], c["head_dim"], bool(c.get("kv_dtype", 0))
    last_loop = c.get("kv_mode", 0) == 1
    caches = {}
    for a, (k, v) in enumerate(cached):
        for inst in range(c["loops"]):
            caches[a, inst] = [case["ctx"] - k.shape[0], _stored(k, fp8), _stored(v, fp8)]

    def slerp(x, o, lr):
        a, b = _justnorm(x), _justnorm(o)
        return _justnorm(a + lr.double() * (b - a))

    def sublayer(l, x, pos0, inst, store):
        L = layers[l]
        if L["kind"] == MLP:
            g = _times(x, L["gate"]) * L["sg"].double()
            h = _justnorm(g * torch.sigmoid(g) * (_times(x, L["up"]) * L["su"].double()))
            return slerp(x, _times(h, L["down"]), L["lr"])
        m, theta = x.shape[0], c["theta_sliding"] if L["kind"] == SLIDING else c["theta_full"]
        q = _justnorm(_rope(_times(x, L["q"]).view(m, heads, d), pos0, theta)) * L["qscale"].double().view(heads, d)
        k = _justnorm(_rope(_times(x, L["k"]).view(m, kv, d), pos0, theta))
        v = _times(x, L["v"]).view(m, kv, d)
        cache = caches[l // 2, inst]
        att = _attend(q, k, v, cache[1], cache[2], pos0, cache[0], c["window"] if L["kind"] == SLIDING else 0)
        if store:
            cache[1], cache[2] = (torch.cat((cache[1], _stored(k, fp8))), torch.cat((cache[2], _stored(v, fp8))))
        gated = _justnorm(att.reshape(m, -1) * torch.sigmoid(_times(x, L["g"]) * L["gscale"].double()))
        return slerp(x, _times(gated, L["o"]), L["lr"])

    for off in range(0, case["m"], 512):
        x = rows[off:off + 512].double()
        pos0 = case["ctx"] + off
        for l in range(c["n_in"]):
            x = sublayer(l, x, pos0, 0, True)
        first = state = x
        for i in range(c["loops"]):
            x = _justnorm(state + first)
            for l in range(c["n_in"], c["n_in"] + c["n_rec"]):
                x = sublayer(l, x, pos0, 0 if last_loop else i, not last_loop or i == c["loops"] - 1)
            state = _justnorm(x)
        x = state
        for l in range(c["n_in"] + c["n_rec"], len(layers)):
            x = sublayer(l, x, pos0, 0, True)
    x = x if case["m"] <= 8 else x[-1:]
    return _times(x, head) * logit_scale.double()


def exact(case, seed):
    kind = case["kind"]
    if kind == "proj":
        ws, x = _proj_inputs(case, seed)
        return torch.cat([_times(x.double(), w).reshape(-1) for w in ws])
    if kind == "head":
        g = _gen(seed)
        w = _bf16_weight(g, case["vocab"], case["k"])
        return _times(_rows(g, case["m"], case["k"], case["x"]).double(), w)
    if kind == "attn":
        kc, vc, q, k, v = _attn_inputs(case, seed)
        p0 = max(0, case["ctx"] - case["window"] - case["n_q"]) if case["window"] else 0
        return _attend(q.double(), k.double(), v.double(), _stored(kc[p0:], case["fp8"]), _stored(vc[p0:], case["fp8"]),
                       case["ctx"], p0, case["window"])
    if kind == "sample":
        return None   # whole numbers
    return _model_exact(case, seed)
