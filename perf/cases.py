"""The framework's work, as cases that can be timed and compared.

Every case goes through the torch front end (powerinfer_x64_amd.runtime) as a serving program
calls it: attention decode and prefill over the paged cache, whole attention and gated-DeltaNet
layer steps, and the TurboQuant compressed cache.  A case is a dict of plain values:

  kind "decode"      attn_decode: one query token a sequence over its cached context
  kind "step"        attn_prologue (norm, RoPE, append) and attn_decode: the attention part of
                     one serving step of a batch
  kind "prefill"     attn_prefill: causal prompts of a batch, contiguous q / k / v
  kind "chunk"       attn_prefill_paged: a chunk of queries over a long cached history
  kind "layer"       AttnLayer: a fresh prompt through norm, RoPE, append, attention, gate
  kind "gdn_layer"   GdnLayer: n tokens through conv, gates, the delta rule and RMSNormGated
  kind "gdn_decode"  gdn_decode: one recurrent step of a batch, states updated in place
  kind "tq"          TqPool.append of n_new tokens a sequence, then tq_attn_decode

Head shapes, contexts and distributions are those of this repository's benchmark and tests:
q, k, v ~ N(0, 1), decay -softplus(N(0, 1)), beta sigmoid(N(0, 1)), pages in random order.
"""
from __future__ import annotations

import math
import random

import torch

from powerinfer_x64_amd import runtime as rt

PAGE = 16
EPS = 1e-6
SECTIONS = (11, 11, 10, 0)  # the sectioned NeoX rotation of the 64 rotary dims
DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_DEV = None


def _dev() -> rt.Device:
    """The program's one library handle."""
    global _DEV
    if _DEV is None:
        _DEV = rt.Device(0)
    return _DEV


# ---- the cases -----------------------------------------------------------------------------

def _attn(kind, name=None, **kw):
    c = {"kind": kind, "hq": 32, "hkv": 8, "d": 128, "dtype": "f16", "gate": False, "norm": False,
         "sections": False, "rope_base": 1e6}
    c.update(kw)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # One chat user on a small f32-cached model: the smallest call, two short launches.
        _attn("decode", "decode_f32_ctx512", hkv=32, dtype="f32", batch=1, ctx_lo=512, ctx_hi=512,
              len_seed=1, rope_base=1e4),
        # A serving batch of ragged long conversations, f16 pages: bound by the cache's bytes.
        _attn("decode", "decode_f16_b32_ragged", batch=32, ctx_lo=1024, ctx_hi=32768, len_seed=2),
        # One step of a batch at 64k context on a gated hybrid-model layer (norm, partial
        # sectioned RoPE, append, attention, gate).
        _attn("step", "step_f16_d256_ctx64k", hq=16, hkv=2, d=256, gate=True, norm=True, sections=True,
              rope_base=1e7, batch=8, ctx_lo=65536, ctx_hi=65536, len_seed=3),
        # One step of a small batch of short, ragged conversations: launches and round trips.
        _attn("step", "step_f16_b4_short", norm=True, batch=4, ctx_lo=100, ctx_hi=3000, len_seed=4),
        # A long prompt on contiguous bf16 rows: the matrix cores' case.
        _attn("prefill", "prefill_bf16_s4096", dtype="bf16", batch=1, s=4096),
        # A batch of odd-length short prompts of a small-head model.
        _attn("prefill", "prefill_f16_d64_b4_s777", d=64, batch=4, s=777),
        # A fresh prompt through a whole gated attention layer with an f16 cache.
        _attn("layer", "layer_f16_d256_n1024", hq=16, hkv=2, d=256, gate=True, norm=True, sections=True,
              rope_base=1e7, n=1024),
        # A fresh odd-length prompt through a layer whose cache keeps full f32 precision.
        _attn("layer", "layer_f32_n1000", hkv=32, dtype="f32", rope_base=1e4, n=1000),
        # A chunk of a long prompt over the history already in the pages (chunked prefill).
        _attn("chunk", "chunk_f16_1000_over_8200", n=1000, hist=8200),
        # A long prompt through a whole gated-DeltaNet layer.
        {"name": "gdn_layer_n4096", "kind": "gdn_layer", "hk": 16, "hv": 32, "n": 4096},
        # One recurrent step of a serving batch: bound by the states' bytes.
        {"name": "gdn_decode_b32", "kind": "gdn_decode", "hk": 16, "hv": 32, "batch": 32},
        # New prompt chunks quantised into the compressed cache, and the decode that follows.
        _attn("tq", "tq_b4_new512", batch=4, ctx_lo=2048, ctx_hi=16384, len_seed=5, n_new=512),
    ]


def _logint(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _heads(rng, d):
    return rng.choice([(16, 2), (8, 2), (16, 4)] if d == 256 else [(32, 8), (32, 32), (8, 4), (12, 4), (16, 2)])


def draw(rng):
    kind = rng.choice(["decode", "decode", "step", "prefill", "prefill", "layer", "layer", "chunk", "gdn_layer",
                       "gdn_layer", "gdn_decode", "tq"])
    if kind == "gdn_layer":
        hk, hv = rng.choice([(16, 32), (16, 32), (2, 4)])
        return {"kind": kind, "hk": hk, "hv": hv, "n": _logint(rng, 1, 4096)}
    if kind == "gdn_decode":
        hk, hv = rng.choice([(16, 32), (16, 32), (2, 4)])
        return {"kind": kind, "hk": hk, "hv": hv, "batch": _logint(rng, 1, 64)}
    d = rng.choice([128, 256] if kind == "tq" else [64, 128, 128, 256])
    hq, hkv = _heads(rng, d)
    norm = rng.random() < 0.5
    kw = {"hq": hq, "hkv": hkv, "d": d, "norm": norm, "sections": norm and d > 64, "rope_base": rng.choice([1e4, 1e6, 1e7]),
          "gate": rng.random() < 0.3 if kind in ("decode", "step", "layer", "tq") else False,
          "dtype": rng.choice(["bf16", "f16"]) if kind == "prefill" else "f16" if kind == "tq" else
          rng.choice(["f16", "f16", "f32"])}
    if kind in ("decode", "step", "tq"):
        c = _attn(kind, **kw, batch=_logint(rng, 1, 32), ctx_lo=_logint(rng, 16, 8192), len_seed=rng.randrange(1 << 20))
        if kind == "tq":
            c["n_new"] = _logint(rng, 1, min(2048, 4096 // c["batch"]))
            c["ctx_lo"] = max(c["ctx_lo"], c["n_new"])
        c["ctx_hi"] = c["ctx_lo"] * rng.randint(1, 8) + rng.randrange(16)
        while sum(_lens(c)) * hkv * 2 * d * (4 if c["dtype"] == "f32" else 2) > 2.0e9:
            c["ctx_hi"] = max(c["ctx_lo"], c["ctx_hi"] // 2)
            c["batch"] = max(1, c["batch"] * 2 // 3)
        return c
    if kind == "prefill":
        c = _attn(kind, **kw, batch=rng.randint(1, 4), s=_logint(rng, 16, 4096))
        while work(c)["flops"] > 1.3e11:
            c["s"] = c["s"] * 3 // 4
        return c
    most = 2e10 if kw["dtype"] == "f32" else 1.3e11
    c = _attn(kind, **kw, n=_logint(rng, 2, 4096 if kind == "layer" else 2048))
    if kind == "chunk":
        c.update(norm=False, sections=False, hist=_logint(rng, 64, 16384))
    while work(c)["flops"] > most:
        c["n"] = max(2, c["n"] * 3 // 4)
    return c


def _lens(c):
    r = random.Random(c["len_seed"])
    return [r.randint(c["ctx_lo"], c["ctx_hi"]) for _ in range(c["batch"])]


def work(case):
    c = case
    if c["kind"] == "gdn_layer":
        n, hk, hv = c["n"], c["hk"], c["hv"]
        conv = 2 * hk * 128 + hv * 128
        # qkv, z, gates in and out once; both states in and out
        b = 4 * (n * (conv + 2 * hv * 128 + 2 * hv) + 2 * 3 * conv + 4 * conv + 2 * hv * 128 * 128)
        return {"bytes": b, "flops": n * hv * 3 * 2 * 128 * 128}
    if c["kind"] == "gdn_decode":
        n, hk, hv = c["batch"], c["hk"], c["hv"]
        return {"bytes": 4 * n * (2 * hk * 128 + 2 * hv * 128 + 2 * hv + 2 * hv * 128 * 128),
                "flops": n * hv * 3 * 2 * 128 * 128}
    hq, hkv, d = c["hq"], c["hkv"], c["d"]
    e = 4 if c["dtype"] == "f32" else 2
    if c["kind"] == "prefill":
        n = c["batch"] * c["s"]
        return {"bytes": n * d * (e * (hq + 2 * hkv) + 4 * hq),
                "flops": 4 * d * hq * c["batch"] * c["s"] * (c["s"] + 1) / 2}
    if c["kind"] == "chunk":
        n, h = c["n"], c["hist"]
        return {"bytes": d * (n * hq * (e + 4) + (h + n) * hkv * 2 * e), "flops": 4 * d * hq * n * (h + (n + 1) / 2)}
    if c["kind"] == "layer":
        n = c["n"]
        # q, k rewritten; v and the gate read; K and V appended; out written
        b = n * d * (4 * (2 * hq + 3 * hkv + hq + (hq if c["gate"] else 0)) + 2 * e * hkv)
        return {"bytes": b, "flops": 4 * d * hq * n * (n + 1) / 2}
    tok, bsz = sum(_lens(c)), c["batch"]
    io = bsz * hq * d * 4 * (3 if c["gate"] else 2)
    flops = 4 * d * hq * tok
    if c["kind"] == "tq":
        new = bsz * c["n_new"] * hkv
        rec = d // 2 + 4 + 2 * d
        return {"bytes": tok * hkv * rec + io + new * (8 * d + rec) + 8 * hkv * d * d, "flops": flops + new * 4 * d * d}
    if c["kind"] == "step":
        io += bsz * d * (4 * (hq + 3 * hkv) + 2 * e * hkv)
    return {"bytes": tok * hkv * 2 * d * e + io, "flops": flops}


def tolerance(case):
    # About four times what the path shows against a 64-bit evaluation of the same inputs
    # (f16 operands 1.3e-4 .. 4e-4, bf16 probabilities 1.3e-3, the f32 paths 4e-7 .. 9e-6,
    # the split-operand delta rule 8e-6 .. 2.4e-5 after its norm, its f32 step 1e-7).
    k = case["kind"]
    if k == "gdn_layer":
        return {"rel": 2e-4}
    if k == "gdn_decode":
        return {"rel": 1e-5}
    if case["dtype"] == "f32":
        return {"rel": 5e-5}
    if k == "prefill":
        return {"rel": 6e-3 if case["dtype"] == "bf16" else 1e-3}
    return {"rel": 2e-3}


# ---- inputs ---------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _kv_dtype(c):
    return DT["f16" if c["dtype"] == "bf16" else c["dtype"]]


def _fill(pool, g, lens, hkv, d, dtype):
    """Random K / V rows of every sequence into the pool; the page table (pages in random order)."""
    pages = [(n + PAGE - 1) // PAGE for n in lens]
    perm = torch.randperm(pool.n_pages, generator=g, device="cuda").to(torch.int32)
    pt = torch.full((len(lens), max(pages)), -1, dtype=torch.int32, device="cuda")
    zero = torch.zeros(1, dtype=torch.int32, device="cuda")
    at = 0
    for i, n in enumerate(lens):
        pt[i, :pages[i]] = perm[at:at + pages[i]]
        at += pages[i]
    for i, n in enumerate(lens):
        k, v = _randn(g, 1, n, hkv, d, dtype=dtype), _randn(g, 1, n, hkv, d, dtype=dtype)
        pool.append(k, v, pt[i:i + 1].contiguous(), zero)
    return pt


def _n_pages(lens):
    return sum((n + PAGE - 1) // PAGE for n in lens)


def _norm_w(g, c):
    """The per-head norm weights and the rotation of the case's layer."""
    if not c["norm"]:
        return None, None
    return tuple(torch.rand((c["d"],), generator=g, device="cuda") + 0.5 for _ in range(2))


def _rope_dim(c):
    return 64 if c["sections"] else c["d"]


def prepare(case, seed):
    c, g, dev = case, _gen(seed), _dev()
    s = {"c": c}
    if c["kind"] == "gdn_decode":
        b, hk, hv = c["batch"], c["hk"], c["hv"]
        s.update(q=_randn(g, b, hk, 128), k=_randn(g, b, hk, 128), v=_randn(g, b, hv, 128),
                 beta=torch.sigmoid(_randn(g, b, hv)), decay=-torch.nn.functional.softplus(_randn(g, b, hv)),
                 state=_randn(g, b, hv, 128, 128) * 0.1, out=torch.empty((b, hv, 128), device="cuda"))
        return s
    if c["kind"] == "gdn_layer":
        x = _gdn_layer_inputs(g, c)
        host = lambda t: t.cpu().numpy()  # noqa: E731
        s["layer"] = rt.GdnLayer(dev, c["hk"], c["hv"], 128, 128, host(x["conv_w"]), host(x["ssm_a"]),
                                 host(x["dt_bias"]), host(x["norm_w"]), EPS)
        s.update(x, out=torch.empty_like(x["z"]))
        return s
    hq, hkv, d, dt = c["hq"], c["hkv"], c["d"], DT[c["dtype"]]
    if c["kind"] == "prefill":
        b, n = c["batch"], c["s"]
        s.update(q=_randn(g, b, n, hq, d, dtype=dt), k=_randn(g, b, n, hkv, d, dtype=dt),
                 v=_randn(g, b, n, hkv, d, dtype=dt), out=torch.empty((b, n, hq, d), device="cuda"))
        return s
    if c["kind"] == "layer":
        n = c["n"]
        wq, wk = _norm_w(g, c)
        s.update(q=_randn(g, n, hq, d), k=_randn(g, n, hkv, d), v=_randn(g, n, hkv, d),
                 gate=_randn(g, n, hq, d) if c["gate"] else None, out=torch.empty((n, hq, d), device="cuda"))
        s["layer"] = rt.AttnLayer(dev, n, hq, hkv, d, _kv_dtype(c), None if wq is None else wq.cpu().numpy(),
                                  None if wk is None else wk.cpu().numpy(), EPS, _rope_dim(c), c["rope_base"],
                                  SECTIONS if c["sections"] else None)
        return s
    if c["kind"] == "chunk":
        lens = [c["hist"] + c["n"]]
        s["pool"] = rt.KvPool(dev, _n_pages(lens), hkv, d, _kv_dtype(c))
        s["row"] = _fill(s["pool"], g, lens, hkv, d, dt)[0].contiguous()
        s.update(q=_randn(g, c["n"], hq, d, dtype=dt), out=torch.empty((c["n"], hq, d), device="cuda"))
        return s
    lens, b = _lens(c), c["batch"]
    if c["kind"] == "tq":
        s["pool"] = rt.TqPool(dev, _n_pages(lens), hkv, d)
        s["pt"] = _fill(s["pool"], g, lens, hkv, d, torch.float32)
        s.update(k=_randn(g, b, c["n_new"], hkv, d), v=_randn(g, b, c["n_new"], hkv, d))
        new = c["n_new"]
    else:
        s["pool"] = rt.KvPool(dev, _n_pages(lens), hkv, d, _kv_dtype(c))
        s["pt"] = _fill(s["pool"], g, lens, hkv, d, dt)
        new = 1
    s["q"] = _randn(g, b, hq, d)
    s["gate"] = _randn(g, b, hq, d) if c["gate"] else None
    s["ctx"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
    s["start"] = s["ctx"] - new
    s["out"] = torch.empty_like(s["q"])
    if c["kind"] == "step":
        s.update(k=_randn(g, b, 1, hkv, d), v=_randn(g, b, 1, hkv, d))
        s["wq"], s["wk"] = _norm_w(g, c)
    return s


def _gdn_layer_inputs(g, c):
    n, hk, hv = c["n"], c["hk"], c["hv"]
    conv = 2 * hk * 128 + hv * 128
    return {"qkv": _randn(g, n, conv), "z": _randn(g, n, hv, 128), "beta_raw": _randn(g, n, hv), "a_raw": _randn(g, n, hv),
            "conv_w": _randn(g, conv, 4) * 0.5, "ssm_a": -torch.rand((hv,), generator=g, device="cuda") - 0.25,
            "dt_bias": _randn(g, hv) * 0.2, "norm_w": torch.rand((128,), generator=g, device="cuda") + 0.5}


# ---- one pass -------------------------------------------------------------------------------

def run(s):
    c, dev = s["c"], _dev()
    kind = c["kind"]
    if kind == "decode":
        return rt.attn_decode(dev, s["q"], s["pool"], s["pt"], s["ctx"], gate=s["gate"], out=s["out"])
    if kind == "step":
        q4 = s["q"].unsqueeze(1)
        rt.attn_prologue(dev, q4, s["k"], s["v"], s["pool"], s["pt"], s["start"], s["wq"], s["wk"], EPS, _rope_dim(c),
                         c["rope_base"], SECTIONS if c["sections"] else None)
        out = rt.attn_decode(dev, s["q"], s["pool"], s["pt"], s["ctx"], gate=s["gate"], out=s["out"])
        return {"out": out, "q": s["q"], "k": s["k"]}
    if kind == "prefill":
        return rt.attn_prefill(dev, s["q"], s["k"], s["v"], out=s["out"])
    if kind == "chunk":
        return rt.attn_prefill_paged(dev, s["q"], s["pool"], s["row"], c["hist"], out=s["out"])
    if kind == "layer":
        s["layer"].reset()  # a new conversation
        out = s["layer"].forward_dev(s["q"], s["k"], s["v"], s["gate"], s["out"])
        return {"out": out, "q": s["q"], "k": s["k"]}
    if kind == "gdn_layer":  # the next n tokens of the layer's sequence
        return s["layer"].forward_dev(s["qkv"], s["z"], s["beta_raw"], s["a_raw"], s["out"])
    if kind == "gdn_decode":
        out = rt.gdn_decode(dev, s["q"], s["k"], s["v"], s["beta"], s["decay"], s["state"], s["out"])
        return {"out": out, "state": s["state"]}
    s["pool"].append(s["k"], s["v"], s["pt"], s["start"])
    return rt.tq_attn_decode(dev, s["q"], s["pool"], s["pt"], s["ctx"], gate=s["gate"], out=s["out"])


# ---- the same in 64 bits --------------------------------------------------------------------

def _attend64(q, k, v, q0):
    """Causal attention of query rows q [n, hq, d] at positions q0 .. over k, v [L, hkv, d], query
    head h reading KV head h % hkv; 64-bit, a block of rows at a time."""
    n, hq, d = q.shape
    total, hkv = k.shape[:2]
    out = torch.empty((n, hq, d), dtype=torch.float64, device=q.device)
    keys = torch.arange(total, device=q.device)
    for j in range(hkv):
        kt, vj = k[:, j].double().t().contiguous(), v[:, j].double().contiguous()
        for h in range(j, hq, hkv):
            for r in range(0, n, 1024):
                m = min(n, r + 1024)
                sc = (q[r:m, h].double() @ kt) / math.sqrt(d)
                if n > 1:
                    at = torch.arange(q0 + r, q0 + m, device=q.device)
                    sc = sc.masked_fill(keys[None] > at[:, None], -math.inf)
                out[r:m, h] = torch.softmax(sc, -1) @ vj
    return out


def _norm_rope64(x, w, pos, c):
    """Per-head RMSNorm (when w) and the rotation of x [n, heads, d] at positions pos [n]."""
    x = x.double()
    if w is not None:
        x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()
    rd = _rope_dim(c)
    i = torch.arange(rd // 2, dtype=torch.float64, device=x.device)
    ang = pos.double()[:, None] * torch.pow(torch.tensor(c["rope_base"], dtype=torch.float64, device=x.device), -2 * i / rd)
    cos, sin = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    y = x.clone()
    a, b = (x[..., :rd // 2], x[..., rd // 2:rd]) if c["sections"] else (x[..., 0:rd:2], x[..., 1:rd:2])
    ra, rb = a * cos - b * sin, a * sin + b * cos
    if c["sections"]:
        y[..., :rd // 2], y[..., rd // 2:rd] = ra, rb
    else:
        y[..., 0:rd:2], y[..., 1:rd:2] = ra, rb
    return y


def _rows(g, c, lens, dt):
    """K / V rows of every sequence as _fill draws them."""
    torch.randperm(_n_pages(lens), generator=g, device="cuda")
    for n in lens:
        yield _randn(g, 1, n, c["hkv"], c["d"], dtype=dt)[0], _randn(g, 1, n, c["hkv"], c["d"], dtype=dt)[0]


def exact(case, seed):
    c, g = case, _gen(seed)
    if c["kind"] == "tq":
        return None  # defined by its stored 3-bit records, not by the attention they approximate
    if c["kind"] == "gdn_decode":
        b, hk, hv = c["batch"], c["hk"], c["hv"]
        q, k, v = _randn(g, b, hk, 128), _randn(g, b, hk, 128), _randn(g, b, hv, 128)
        beta, decay = torch.sigmoid(_randn(g, b, hv)), -torch.nn.functional.softplus(_randn(g, b, hv))
        st = (_randn(g, b, hv, 128, 128) * 0.1).double()
        out = _delta64(q, k, v.double(), beta.double(), decay.double(), st, hk, hv)
        return {"out": out, "state": st}
    if c["kind"] == "gdn_layer":
        return _gdn_layer64(c, _gdn_layer_inputs(g, c))
    hq, hkv, d, dt = c["hq"], c["hkv"], c["d"], DT[c["dtype"]]
    if c["kind"] == "prefill":
        b, n = c["batch"], c["s"]
        q, k, v = (_randn(g, b, n, h, d, dtype=dt) for h in (hq, hkv, hkv))
        return torch.stack([_attend64(q[i], k[i], v[i], 0) for i in range(b)])
    if c["kind"] == "layer":
        n = c["n"]
        wq, wk = _norm_w(g, c)
        q, k, v = (_randn(g, n, h, d) for h in (hq, hkv, hkv))
        pos = torch.arange(n, device="cuda")
        qr, kr = _norm_rope64(q, wq, pos, c), _norm_rope64(k, wk, pos, c)
        out = _attend64(qr, kr, v, 0)
        return {"out": out * torch.sigmoid(_randn(g, n, hq, d).double()) if c["gate"] else out, "q": qr, "k": kr}
    if c["kind"] == "chunk":
        (k, v), = _rows(g, c, [c["hist"] + c["n"]], dt)
        return _attend64(_randn(g, c["n"], hq, d, dtype=dt), k, v, c["hist"])
    lens, b = _lens(c), c["batch"]
    kept = list(_rows(g, c, lens, dt))
    q = _randn(g, b, hq, d)
    gate = torch.sigmoid(_randn(g, b, hq, d).double()) if c["gate"] else 1.0
    k_new = None
    if c["kind"] == "step":
        k_new, v_new = _randn(g, b, 1, hkv, d)[:, 0], _randn(g, b, 1, hkv, d)[:, 0]
        wq, wk = _norm_w(g, c)
        pos = torch.tensor(lens, device="cuda") - 1
        q, k_new = _norm_rope64(q, wq, pos, c), _norm_rope64(k_new, wk, pos, c)
    out = torch.empty((b, hq, d), dtype=torch.float64, device="cuda")
    for i, (k, v) in enumerate(kept):
        if k_new is not None:
            k, v = (torch.cat([t[:-1].double(), x[i:i + 1].double()]) for t, x in ((k, k_new), (v, v_new)))
        out[i:i + 1] = _attend64(q[i:i + 1], k, v, lens[i] - 1)
    out = out * gate
    return out if k_new is None else {"out": out, "q": q, "k": k_new[:, None]}


def _unit(x):
    return x / torch.clamp(x.norm(dim=-1, keepdim=True), min=1e-12)


def _delta64(q, k, v, beta, decay, st, hk, hv):
    """One step of the delta rule on st [b, hv, 128, 128] (in place); V head h reads K head h % hk."""
    tile = lambda x: _unit(x.double()).repeat(1, hv // hk, 1)  # noqa: E731
    qh, kh = tile(q) / math.sqrt(128), tile(k)
    st *= torch.exp(decay)[..., None, None]
    delta = (v - (st * kh[..., None]).sum(-2)) * beta[..., None]
    st += kh[..., None] * delta[..., None, :]
    return (st * qh[..., None]).sum(-2)


def _gdn_layer64(c, x):
    """The layer's n tokens from a fresh state, token by token."""
    n, hk, hv = c["n"], c["hk"], c["hv"]
    ext = torch.cat([torch.zeros((3, x["qkv"].shape[1]), dtype=torch.float64, device="cuda"), x["qkv"].double()])
    w = x["conv_w"].double()
    act = sum(ext[j:j + n] * w[:, j] for j in range(4))
    act = act * torch.sigmoid(act)
    q, k, v = act.split([hk * 128, hk * 128, hv * 128], dim=1)
    q, k, v = q.view(n, hk, 128), k.view(n, hk, 128), v.view(n, hv, 128)
    beta = torch.sigmoid(x["beta_raw"].double())
    decay = x["ssm_a"].double() * torch.nn.functional.softplus(x["a_raw"].double() + x["dt_bias"].double())
    st = torch.zeros((1, hv, 128, 128), dtype=torch.float64, device="cuda")
    o = torch.empty((n, hv, 128), dtype=torch.float64, device="cuda")
    for t in range(n):
        o[t] = _delta64(q[t:t + 1], k[t:t + 1], v[t:t + 1], beta[t:t + 1], decay[t:t + 1], st, hk, hv)[0]
    z = x["z"].double()
    return o / torch.sqrt((o * o).mean(-1, keepdim=True) + EPS) * x["norm_w"].double() * z * torch.sigmoid(z)
