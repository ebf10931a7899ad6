"""The weaker conditions that settle a controlled row's token where the plain
margins fail (order_settled's runs, draw_refined in xs_sampler.hip), tested by
brute force on the CPU oracle as test_settle_model.py tests the plain ones:
wherever the restated conditions pass, every denominator D within the serial
sum's error bound draws the token that S draws.

Rows hold pairs and triples of logits one to three ulps apart, their ids in
both orders, near the top and around the top-k boundary; uniforms are packed
around every cumulative-weight boundary, and top_p lies on prefix sums, so the
cut is ambiguous too."""
import numpy as np
import pytest

from tests import workloads
from tests.test_settle_model import NEG, _chain, _f32

UU = 2.0 ** -23 * 1.02


def _cut(c, k, top_p):
    for j in range(k):
        if c[j] >= np.float32(top_p):
            return j + 1, True
    return k, False


def _refined(c, w, u, idx, keep, k, found, renorm, S, top_p):
    """draw_refined, restated: c the prefix sums of all k weights, w the weights."""
    sl = (2.0 * k + 8.0) * 2.0 ** -148 * S + 2.0 ** -50
    u = float(u)

    def draw(kept, total):
        x = float(np.float32(u) * np.float32(total))
        n = sum(1 for j in range(k - 1) if (float(c[j]) if j < kept - 1 else total) <= x)

        def m(j):
            cj = float(c[j])
            B = 2 * ((1 - u) * cj + u * (total - cj)) + (1 - u) * j * cj + u * (kept - 1 - j) * total + 2 * u * total
            return UU * B + sl
        ok = n == idx
        if idx >= 1:
            ok = ok and x - float(c[idx - 1]) > m(idx - 1)
        if idx < kept - 1:
            ok = ok and float(c[idx]) - x > m(idx)
        return ok

    def mc(j, cj):
        return UU * (k + j + 4) * cj + sl
    tot = float(c[keep - 1])
    if not draw(keep, tot):
        return False
    if not renorm:
        return True
    tp = float(np.float32(top_p))
    if not found:
        return k < 2 or tp - float(c[k - 2]) > mc(k - 2, float(c[k - 2]))
    if not tot - tp > mc(keep - 1, tot) and keep < k:
        t2 = float(np.float32(tot) + w[keep])
        if not t2 - tp > mc(keep, t2) or not draw(keep + 1, t2):
            return False
    if keep >= 2:
        c1 = float(c[keep - 2])
        if not tp - c1 > mc(keep - 2, c1):
            if keep >= 3 and not tp - float(c[keep - 3]) > mc(keep - 3, float(c[keep - 3])):
                return False
            if not draw(keep - 1, c1):
                return False
    return True


def _ambiguous(e, ids, k, S, enc, e_below):
    """order_settled's positions: e and ids of the selection in logit order."""
    thr = S * (1.01 + enc * 2.0 ** -24 * 1.02) * 2.0 ** -148

    def robust(a, b):
        g = float(a) - float(b)
        return a == b or (g > 2.0 ** -21 * float(a) and g > thr)
    amb, start, op, desc = set(), 0, False, False
    n = len(e)
    for i in range(n):
        link = False
        if i + 1 < n:
            rob = robust(e[i], e[i + 1])
            link = e[i] == e[i + 1] or not rob
            if link:
                op |= not rob and float(e[i]) >= NEG
                desc |= ids[i] > ids[i + 1]
        if not link:
            if i == n - 1:
                desc |= not (e_below < e[i] and robust(e[i], e_below))
            if op and desc:
                amb |= set(range(start, i + 1))
            start, op, desc = i + 1, False, False
    return amb


@pytest.mark.parametrize("seed", range(6))
def test_refined_settlement_is_denominator_free(oracle, seed):
    rng = np.random.default_rng(7700 + seed)
    v, k = 2048, [2, 5, 12, 20, 20, 40][seed]
    T = [1.0, 0.7, 1.0, 1.3, 1.0, 0.7][seed]
    x = rng.normal(0, 2.0, v).astype(np.float32)
    top = np.sort(rng.uniform(4, 8, k + 3).astype(np.float32))[::-1]
    spots = rng.permutation(v)[:k + 3]
    x[spots] = top
    for _ in range(max(2, k // 3)):  # near-ties: one entry a few ulps below another, ids either way
        i = int(rng.integers(0, k + 1))
        t = x[spots[i]]
        for _ in range(int(rng.integers(1, 4))):
            t = np.nextafter(t, np.float32(-np.inf))
        x[spots[i + 1]] = t
    allow = rng.random(v) < 0.5
    allow[spots] = True
    mask = workloads.pack_mask(allow[None, :])[0]
    ctl = oracle.Ctl(allowed=mask)
    vals = np.where(allow, x, -np.inf).astype(np.float32)
    s = (vals * _f32(1.0 / T)).astype(np.float32) if T != 1.0 else vals
    order = np.lexsort((np.arange(v), -vals))
    sel = order[:k + 1]
    e_all = np.array([oracle.exp(float(_f32(s[i] - s.max()))) for i in order[:k + 2]], np.float32)
    e = e_all[:k + 1]
    base = dict(ctl=ctl)
    o64 = oracle.sample_controlled(x, v, T, k, 1.0, u=0.0, sum_mode=oracle.SUM_F64, **base)
    oseq = oracle.sample_controlled(x, v, T, k, 1.0, u=0.0, sum_mode=oracle.SUM_SEQ_F32, **base)
    S = np.float32(o64.ssum)
    delta = v * 2.0 ** -24
    Ds = [np.float32(oseq.ssum)] + [np.float32(float(S) * (1.0 + f * delta)) for f in rng.uniform(-1, 1, 24)]
    amb = _ambiguous(e, [int(i) for i in sel], k, float(S), v, float(e_all[k + 1]))
    # the weights S gives, and top_p on and next to their prefix sums
    p = np.sort((e[:k] / S).astype(np.float32))[::-1]
    sumc = np.float32(-0.0)
    for t in p:
        sumc = np.float32(sumc + t)
    w = (p / sumc).astype(np.float32)
    c = _chain(w)
    at = c[int(rng.integers(0, max(1, k - 1)))]
    settled = refused = 0
    for top_p in [1.0, 0.95, float(at), float(np.nextafter(at, np.float32(2))), float(np.nextafter(at, np.float32(0)))]:
        renorm = np.float32(top_p) < 1.0
        cc, ww = (c, w) if renorm else (_chain(p), p)
        keep, found = _cut(cc, k, top_p) if renorm else (k, False)
        tot = cc[keep - 1]
        us = list(rng.random(30).astype(np.float32))
        for j in range(keep - 1):
            b = float(cc[j]) / float(tot)
            us += [np.float32(min(max(b + d * 2.0 ** -24, 0.0), 1 - 2.0 ** -24))
                   for d in list(range(-8, 9, 2)) + [-60, -25, 25, 60]]
        for u in us:
            xd = np.float32(np.float32(u) * tot)
            idx = sum(1 for j in range(k - 1) if (cc[j] if j < keep - 1 else tot) <= xd)
            if idx in amb or not _refined(cc, ww, u, idx, keep, k, found, renorm, float(S), top_p):
                refused += 1
                continue
            settled += 1
            toks = {oracle.sample_controlled(x, v, T, k, top_p, u=float(u), sum_mode=oracle.SUM_GIVEN,
                                             s_given=float(D), **base).token for D in [S] + Ds}
            assert len(toks) == 1, (seed, top_p, float(u), idx, toks)
    assert settled > 100 and refused > 0, (settled, refused)
