"""The calls whose speed is watched: what one engine step asks of the sampler.

A case is one call through a public entry point: the C ABI of include/xsamp.h
(xs_sample, xs_verify, xs_argmax_probs), called as an engine calls it, with the
argument struct, the context and the device buffers it keeps between steps, or
the Python Sampler.  Logits are what a language model's head leaves (a bulk of
normal or heavy-tailed values with a few tall tokens); vocabulary 248,320 and
the options are the configurations bench.py and the tests name, the other sizes
are generic.

Kinds: "sample" (xs_sample, with whatever the case's options ask for), "verify"
(a speculative block), "argmax" (the drafter's confidence), "sampler" (the
Python Sampler, host uniforms in, host ids out).
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from xwen_amd import _lib
from xwen_amd import sampler as xsm

V = 248_320
WHOLE = 2**31 - 1  # a top_k at or past the vocabulary: top-p only

# Every option a case may set, at the value that leaves it out.
DEFAULTS = dict(kind="sample", rows=1, vocab=V, temperature=1.0, top_k=20, top_p=0.95, sd=3.0, heavy=False,
                mixed=False, masked=False, control=0, cand=0, sums=False, n_top=0, n_score=0, n_class=0,
                span=1)


def listed() -> list[dict]:
    return [
        # One user's decode step, thinking defaults, with the top-20 weights.
        dict(name="one_row", rows=1, cand=20),
        # The smallest call: one greedy row of a small, odd vocabulary.
        dict(name="small_greedy", rows=1, vocab=32_003, temperature=0.0),
        # The Python mirror, a few requests: host uniforms in, host ids out.
        dict(name="python_sampler", kind="sampler", rows=4, temperature=0.7, top_p=0.80),
        # A part-filled, grammar-constrained batch at a wider top_k, on a smaller
        # vocabulary that is no multiple of anything.
        dict(name="ragged_masked24", rows=24, vocab=64_003, temperature=0.8, top_k=50, top_p=0.90, masked=True),
        # The headline: a serving batch with instruct defaults and the top-20 (id, weight).
        dict(name="batch64", rows=64, temperature=0.7, top_p=0.80, sd=2.5, cand=20),
        # Grammar-constrained requests: an allow-mask per row.
        dict(name="masked32", rows=32, masked=True),
        # The same at top_p 1 (a client's default) with candidate weights: the
        # reference's serial denominator reaches the caller.
        dict(name="masked_weights32", rows=32, masked=True, top_p=1.0, cand=20, sums=True),
        # Thinking-budget and penalty controls: bans, biases and a pull per row.
        dict(name="controls16", rows=16, control=300),
        # A speculative verify block, 16 sequences of 15 drafts and the bonus row.
        dict(name="verify16x16", kind="verify", rows=256, span=16),
        # A large batch of different requests, each with log-probs of its best ids.
        dict(name="hetero256", rows=256, mixed=True, heavy=True, n_top=20),
        # Top-p only (no top_k) over a serving batch, tokens.
        dict(name="top_p_only64", rows=64, temperature=0.7, top_k=WHOLE, top_p=0.80, sd=2.5),
        # Scoring held rows: log-probs of listed ids and the masses of two classes.
        dict(name="score16", rows=16, temperature=0.0, n_top=5, n_score=32, n_class=2),
    ]


def draw(rng) -> dict:
    """One more case of those ranges."""
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def vocab():
        return V if rng.random() < 0.3 else logint(16_384, 262_144)

    temperature, top_p = rng.choice([0.6, 0.7, 1.0, 1.3]), rng.choice([0.8, 0.9, 0.95, 1.0])
    c = dict(rows=logint(1, 256), vocab=vocab(), temperature=temperature, top_p=top_p,
             top_k=rng.choice([5, 20, 40, 50, 100]), sd=rng.choice([2.0, 2.5, 3.0]))
    what = rng.choice(["plain", "plain", "masked", "weights", "control", "verify", "mixed", "wide", "score",
                       "argmax", "sampler", "greedy"])
    if what == "plain":
        c["cand"] = rng.choice([0, c["top_k"]])
    elif what == "greedy":
        c.update(temperature=0.0, n_top=rng.choice([0, 1, 20]))
    elif what == "masked":
        c.update(rows=logint(1, 128), masked=True)
    elif what == "weights":
        c.update(rows=logint(1, 64), masked=True, top_p=1.0, cand=c["top_k"], sums=True)
    elif what == "control":
        c.update(rows=logint(1, 64), control=logint(4, 1000), masked=rng.random() < 0.3)
    elif what == "verify":
        span = rng.randint(2, 16)
        c.update(kind="verify", span=span, rows=span * logint(1, 16), masked=rng.random() < 0.3)
    elif what == "mixed":
        c.update(mixed=True, heavy=rng.random() < 0.5, n_top=rng.choice([0, 5, 20]))
    elif what == "wide":
        whole = rng.random() < 0.6
        c.update(rows=logint(1, 32 if whole else 8), top_k=WHOLE if whole else logint(128, 2000))
        c["cand"] = 0 if whole else rng.choice([0, c["top_k"]])
    elif what == "score":
        c.update(rows=logint(1, 64), temperature=0.0, n_top=rng.choice([0, 5]), n_score=logint(1, 256),
                 n_class=rng.randint(0, 3))
    elif what == "argmax":
        c.update(kind="argmax", rows=logint(1, 64))
    elif what == "sampler":
        c.update(kind="sampler", rows=logint(1, 16))
    return c


# ---------------------------------------------------------------------------
# Inputs


def _options(c, rng):
    """Per-row (temperature, top_k, top_p)."""
    n = c["rows"]
    if c["mixed"]:
        return (rng.choice([0.0, 0.6, 0.7, 1.0, 1.3], n), rng.choice([1, 20, 50, 100], n),
                rng.choice([0.8, 0.95, 1.0], n))
    return np.full(n, c["temperature"]), np.full(n, c["top_k"], np.int64), np.full(n, c["top_p"])


def _logits(c, g):
    """[rows, ld] float32: the bulk, then 8 tall tokens a row; the columns past
    the encodable ids hold whatever the head's padding holds."""
    n, enc = c["rows"], c["vocab"]
    ld = (enc + 3) // 4 * 4
    x = torch.randn((n, ld), generator=g, device="cuda")
    if c["heavy"]:  # Student-t(3) x 2
        chi = torch.zeros_like(x)
        for _ in range(3):
            chi += torch.randn((n, ld), generator=g, device="cuda").square_()
        x = x / (chi / 3.0).sqrt_() * 2.0
    else:
        x *= c["sd"]
        at = torch.randint(0, enc, (n, 8), generator=g, device="cuda")
        x.scatter_(1, at, torch.rand((n, 8), generator=g, device="cuda") * 6.0 + 8.0)
    return x


def _pack(allow):
    """bool [..., enc] -> int32 words, bit t % 32 of word t / 32."""
    enc = allow.shape[-1]
    words = (enc + 31) // 32
    pad = torch.zeros((*allow.shape[:-1], words * 32), dtype=torch.int64, device=allow.device)
    pad[..., :enc] = allow
    w = (pad.view(*allow.shape[:-1], words, 32) << torch.arange(32, device=allow.device)).sum(-1)
    return torch.where(w >= 2**31, w - 2**32, w).to(torch.int32).contiguous()


def _mask(c, g, rng):
    """Allow-masks: by thirds a few ranges (about 1 %), 10 % and 50 % of the ids."""
    n, enc = c["rows"], c["vocab"]
    allow = torch.rand((n, enc), generator=g, device="cuda")
    allow = allow < torch.tensor([(0.0, 0.1, 0.5)[r % 3] for r in range(n)], device="cuda")[:, None]
    for r in range(0, n, 3):
        for _ in range(4):
            start = int(rng.integers(0, enc - enc // 400))
            allow[r, start:start + enc // 400] = True
    return allow


def _controls(c, x, rng):
    """Per row: two thirds of the list bans, a third biases, every other row a pull."""
    out = []
    top = x[:, :c["vocab"]].argmax(1).cpu().numpy()
    for r in range(c["rows"]):
        ids = rng.integers(0, c["vocab"], c["control"])
        nb = 2 * c["control"] // 3
        banned = [int(top[r])] + [int(i) for i in ids[:nb]]
        bias = [(int(i), float(np.float32(d))) for i, d in zip(ids[nb:], rng.normal(0, 2, len(ids) - nb))]
        pull = (int(rng.integers(0, c["vocab"])), 0.5) if r % 2 else None
        out.append(xsm.SampleControl(banned=tuple(banned), bias=tuple(bias), pull=pull))
    return out


def _inputs(case, seed):
    """What prepare and exact start from: everything a call reads."""
    c = {**DEFAULTS, **case}
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    rng = np.random.default_rng(seed)
    s = {"c": c, "x": _logits(c, g), "options": _options(c, rng),
         "u": (rng.integers(0, 1 << 23, c["rows"]) * 2.0**-23).astype(np.float32)}
    if c["masked"]:
        s["allow"] = _mask(c, g, rng)
    if c["control"]:
        s["controls"] = _controls(c, s["x"], rng)
    if c["n_score"]:
        s["score_ids"] = torch.as_tensor(rng.integers(0, c["vocab"], (c["rows"], c["n_score"])).astype(np.int32)).cuda()
    if c["n_class"]:
        share = torch.tensor([0.02, 0.5, 0.9][:c["n_class"]], device="cuda")[None, :, None]
        s["classes"] = torch.rand((c["rows"], c["n_class"], c["vocab"]), generator=g, device="cuda") < share
    if c["kind"] == "verify":  # half the drafts the row's argmax, half random
        best = s["x"][:, :c["vocab"]].argmax(1).cpu().numpy().reshape(-1, c["span"])[:, :-1]
        other = rng.integers(0, c["vocab"], best.shape)
        s["drafts"] = np.where(rng.random(best.shape) < 0.5, best, other).astype(np.int32)
    return s


# ---------------------------------------------------------------------------
# One call


def _ptr(a, field, t):
    setattr(a, field, t.data_ptr())
    return t


def prepare(case, seed):
    s = _inputs(case, seed)
    c, x = s["c"], s["x"]
    rows, ld = x.shape
    enc = c["vocab"]
    t, k, p = s["options"]
    if c["kind"] == "sampler":
        opts = xsm.SamplerOptions(temperature=c["temperature"], top_k=c["top_k"], top_p=c["top_p"])
        return {"c": c, "x": x[:, :enc].contiguous(), "u": s["u"],
                "sampler": xsm.Sampler(opts, [enc - 1], enc, max_rows=rows)}
    ctx = xsm.Context(max_rows=rows, vocab=enc, k_max=max(127, int(min(np.max(k), enc))))
    ctx.bind_current_stream()
    lib = _lib.load()
    keep = [ctx, x]
    out = {}

    def new(a, field, shape, dtype):
        out[field] = _ptr(a, field, torch.zeros(shape, dtype=dtype, device="cuda"))

    i32, f32, f64 = torch.int32, torch.float32, torch.float64
    if c["kind"] == "argmax":
        a = _lib.ArgmaxArgs()
        a.logits, a.rows, a.ld, a.width = x.data_ptr(), rows, ld, enc
        new(a, "ids", rows, i32)
        new(a, "probs", rows, f32)
        return {"c": c, "call": lib.xs_argmax_probs, "h": ctx.h, "args": C.byref(a), "out": out, "keep": keep}
    a = _lib.VerifyArgs() if c["kind"] == "verify" else _lib.SampleArgs()
    a.logits, a.ld, a.width, a.enc = x.data_ptr(), ld, ld, enc
    keep.append(_ptr(a, "params", xsm.params_tensor(t, k, p, rows, x.device)))
    keep.append(_ptr(a, "uniforms", torch.as_tensor(s["u"]).cuda()))
    if c["masked"]:
        w = _ptr(a, "allowed", _pack(s["allow"]))
        a.allowed_words = a.allowed_ld = w.shape[1]
        keep.append(w)
    if c["control"]:
        ctl = xsm.controls_tensor(s["controls"], x.device)
        keep += [_ptr(a, "controls", ctl.rows), _ptr(a, "ctl_ids", ctl.ids), _ptr(a, "ctl_delta", ctl.delta)]
    if c["kind"] == "verify":
        a.seqs, a.span = rows // c["span"], c["span"]
        keep.append(_ptr(a, "drafts", torch.as_tensor(s["drafts"]).cuda()))
        for f in ("row_token", "row_status"):
            new(a, f, rows, i32)
        for f in ("accepted", "n_committed", "seq_status"):
            new(a, f, a.seqs, i32)
        new(a, "committed", (a.seqs, a.span), i32)
        return {"c": c, "call": lib.xs_verify, "h": ctx.h, "args": C.byref(a), "out": out, "keep": keep}
    a.rows = rows
    new(a, "token", rows, i32)
    new(a, "status", rows, i32)
    if c["cand"]:
        a.cand_ld = c["cand"]
        new(a, "cand_id", (rows, c["cand"]), i32)
        new(a, "cand_w", (rows, c["cand"]), f32)
        new(a, "n_cand", rows, i32)
    if c["sums"]:
        new(a, "soft_max", rows, f32)
        new(a, "soft_sum", rows, f32)
    if c["n_top"] or c["n_score"]:
        new(a, "row_max", rows, f32)
        new(a, "row_lse", rows, f64)
    if c["n_top"]:
        a.n_top = a.top_ld = c["n_top"]
        new(a, "top_id", (rows, c["n_top"]), i32)
        new(a, "top_logprob", (rows, c["n_top"]), f32)
    if c["n_score"]:
        a.n_score = a.score_ld = c["n_score"]
        keep.append(_ptr(a, "score_ids", s["score_ids"]))
        new(a, "score_logprob", (rows, c["n_score"]), f64)
    if c["n_class"]:
        w = _ptr(a, "class_masks", _pack(s["classes"]))
        a.n_class, a.class_ld = c["n_class"], w.shape[-1]
        keep.append(w)
        new(a, "class_mass", (rows, c["n_class"]), f64)
    if c["mixed"]:  # a batch of different requests starts its costliest rows first
        order = xsm.cost_order(t, k)
        a.row_order = order.ctypes.data
        keep.append(order)
    return {"c": c, "call": lib.xs_sample, "h": ctx.h, "args": C.byref(a), "out": out, "keep": keep}


def run(state):
    if state["c"]["kind"] == "sampler":
        return state["sampler"].sample(state["x"], state["u"])
    rc = state["call"](state["h"], state["args"])
    if rc:
        raise RuntimeError(f"call failed: {rc}")
    return state["out"]


def work(case):
    """Each logit, mask word and listed id read once, each output written once;
    an operation count of a few per logit (scale, subtract, exp, add)."""
    c = {**DEFAULTS, **case}
    n, enc, words = c["rows"], c["vocab"], (c["vocab"] + 31) // 32
    b = 4.0 * n * enc + 28.0 * n
    if c["masked"]:
        b += 4.0 * n * words
    b += n * (8.0 * c["cand"] + 12.0 * c["control"] + 8.0 * c["n_top"] + 12.0 * c["n_score"])
    b += n * c["n_class"] * (4.0 * words + 8.0)
    return {"bytes": b, "flops": 4.0 * n * enc}


def tolerance(case):
    """Ids are whole.  Weights, sums and log-probs are 32-bit sums and exps."""
    return {"rel": 1.6e-6, "max": 2e-5}


# ---------------------------------------------------------------------------
# The same in 64 bits


def exact(case, seed):
    s = _inputs(case, seed)
    c = s["c"]
    n, enc = c["rows"], c["vocab"]
    if c["kind"] in ("sampler", "verify"):
        return None  # whole numbers only
    x = s["x"][:, :enc].double()
    t, k, p = s["options"]
    if c["kind"] == "argmax":
        return {"ids": x.argmax(1).int(), "probs": 1.0 / (x - x.max(1, keepdim=True).values).exp().sum(1)}
    out = {}
    if c["n_top"] or c["n_score"]:
        lse = torch.logsumexp(x, 1)
        out.update(row_max=x.max(1).values, row_lse=lse)
        if c["n_top"]:
            v, i = x.sort(dim=1, descending=True, stable=True)
            out.update(top_id=i[:, :c["n_top"]].int(), top_logprob=v[:, :c["n_top"]] - lse[:, None])
        if c["n_score"]:
            out["score_logprob"] = x.gather(1, s["score_ids"].long()) - lse[:, None]
        if c["n_class"]:
            q = (x - lse[:, None]).exp()
            out["class_mass"] = torch.stack([(q * s["classes"][:, j]).sum(1) for j in range(c["n_class"])], 1)
    if (c["cand"] or c["sums"]) and not c["mixed"]:
        if c["masked"]:
            x = x.masked_fill(~s["allow"], -math.inf)
        z = x / c["temperature"]
        m = z.max(1).values
        e = (z - m[:, None]).exp()
        if c["sums"]:
            out.update(soft_max=m, soft_sum=e.sum(1))
        if c["cand"]:
            w = e / e.sum(1, keepdim=True)
            w, i = w.sort(dim=1, descending=True, stable=True)
            w = w[:, :c["cand"]]
            if c["top_p"] < 1.0:
                w = w / w.sum(1, keepdim=True)
                before = w.cumsum(1) - w
                w = torch.where(before >= float(np.float32(c["top_p"])), 0.0, w)
            out.update(cand_id=i[:, :c["cand"]].int(), cand_w=w)
    return out or None
