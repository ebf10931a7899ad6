"""When a controlled row is left to the serial sum: the finalizer's own decision,
row by row, on rows made to sit on it.

A masked row of a call that takes tokens only is settled by the plain margins,
by the weaker conditions (a run of near-equal entries whose order cannot change
the drawn id, the draw's own margins, the cut on either side of top_p), or is
summed serially and counted (xs_test_serial_fallback).  The rows here hold
pairs of logits one to three ulps apart with ids in both orders, pairs that
straddle list positions 63 and 64 and the top-k edge among them, draw from
uniforms packed around the cumulative-weight boundaries, and put top_p on
prefix sums.  top_k up to 63 takes the fast finalizer, above it the general one.

Every token must be the serial-f32 reference's, and every row must be sent to
the serial sum exactly when the conditions, restated here, say so."""
import ctypes

import numpy as np
import pytest

from tests import workloads
from tests.test_gpu_sampler import run_sample
from tests.test_settle_model import NEG, _chain

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _plain(c, u, idx, keep, k, found, renorm, S, top_p, f):
    """draw_settled, its margins times f."""
    uu = f * 2.0 ** -23 * 1.02
    sl = f * ((2.0 * k + 8.0) * 2.0 ** -148 * S + 2.0 ** -50)

    def m(j):
        return uu * (k + j + 4) * float(c[j])
    tot, tp = c[keep - 1], float(np.float32(top_p))
    x = float(np.float32(u) * tot)
    ok = True
    if renorm and found:
        ok = float(tot) - tp > m(keep - 1) + sl
        if keep >= 2:
            ok = ok and tp - float(c[keep - 2]) > m(keep - 2) + sl
    elif renorm:
        ok = tp - float(c[k - 1]) > m(k - 1) + sl
    mt = uu * (k + keep + 4) * float(tot) + sl
    if idx >= 1:
        ok = ok and x - float(c[idx - 1]) > m(idx - 1) + mt
    if idx < keep - 1:
        ok = ok and float(c[idx]) - x > m(idx) + mt
    return ok


def _refined(c, w, u, idx, keep, k, found, renorm, S, top_p, f):
    """draw_refined, its margins times f."""
    uu = f * 2.0 ** -23 * 1.02
    sl = f * ((2.0 * k + 8.0) * 2.0 ** -148 * S + 2.0 ** -50)
    u, tp = float(u), float(np.float32(top_p))

    def draw(kept, total):
        total = np.float32(total)
        x = float(np.float32(u) * total)
        total = float(total)
        n = sum(1 for j in range(k - 1) if (float(c[j]) if j < kept - 1 else total) <= x)

        def m(j):
            cj = float(c[j])
            return uu * (2 * ((1 - u) * cj + u * (total - cj)) + (1 - u) * j * cj + u * (kept - 1 - j) * total
                         + 2 * u * total) + sl
        ok = n == idx
        if idx >= 1:
            ok = ok and x - float(c[idx - 1]) > m(idx - 1)
        if idx < kept - 1:
            ok = ok and float(c[idx]) - x > m(idx)
        return ok

    def mc(j, cj):
        return uu * (k + j + 4) * cj + sl
    tot = float(c[keep - 1])
    if not draw(keep, tot):
        return False
    if not renorm:
        return True
    if not found:
        return k < 2 or tp - float(c[k - 2]) > mc(k - 2, float(c[k - 2]))
    if not tot - tp > mc(keep - 1, tot) and keep < k:
        t2 = float(np.float32(tot) + w[keep])
        if not t2 - tp > mc(keep, t2) or not draw(keep + 1, t2):
            return False
    if keep >= 2 and not tp - float(c[keep - 2]) > mc(keep - 2, float(c[keep - 2])):
        if keep >= 3 and not tp - float(c[keep - 3]) > mc(keep - 3, float(c[keep - 3])):
            return False
        return draw(keep - 1, float(c[keep - 2]))
    return True


def _order(e, ids, k, S, enc, below):
    """order_settled over a selection of k + 1 in logit order: whether it fails
    whatever is drawn, whether the plain condition holds, and the positions the
    denominator may reorder.  below: the largest e outside the selection."""
    thr = S * (1.01 + enc * 2.0 ** -24 * 1.02) * 2.0 ** -148
    n = len(e)

    def robust(a, b):
        g = float(a) - float(b)
        return a == b or (g > 2.0 ** -21 * float(a) and g > thr)
    fails = e[k - 1] == e[-1] and e[k - 1] >= NEG and not (below < e[-1] and robust(e[-1], below))
    plain = all(robust(e[i], e[i + 1]) for i in range(n - 1) if e[i] >= NEG)
    amb, start, loose, desc = set(), 0, False, False
    for i in range(n):
        link = i + 1 < n and (e[i] == e[i + 1] or not robust(e[i], e[i + 1]))
        if link:
            loose |= not robust(e[i], e[i + 1]) and e[i] >= NEG
            desc |= ids[i] > ids[i + 1]
            continue
        if i == n - 1:
            desc |= not (below < e[i] and robust(e[i], below))
        if loose and desc:
            amb |= set(range(start, i + 1))
        start, loose, desc = i + 1, False, False
    return bool(fails), plain and not fails, amb


def _row(rng, v, k, scale):
    """Logits with k + 3 tall values, some of them one to three ulps below their
    predecessor (one pair at positions 63 and 64, one at the top-k edge)."""
    x = rng.normal(-9 * scale, scale, v).astype(np.float32)
    top = np.sort(rng.uniform(-0.2 * scale, 2.0 * scale, k + 3).astype(np.float32))[::-1].copy()
    at = {int(i) for i in rng.integers(0, k + 1, max(2, k // 12))}
    at |= {int(i) for i in (62, 63, k - 2, k - 1) if 0 <= i <= k and rng.random() < (0.8 if i < k - 2 else 0.3)}
    for i in sorted(at):
        top[i + 1] = top[i]
        for _ in range(int(rng.integers(1, 4))):
            top[i + 1] = np.nextafter(top[i + 1], np.float32(-np.inf))
    top = np.sort(top)[::-1]
    spots = rng.permutation(v)[:k + 3]
    if rng.random() < 0.4:  # (every run's ids ascend)
        spots = np.sort(spots)
    x[spots] = top
    allow = rng.random(v) < 0.5
    allow[spots] = True
    return x, allow, sorted(at)


@pytest.mark.parametrize("v,k,rows", [(4_096, 5, 40), (4_096, 20, 40), (70_000, 20, 16), (4_096, 62, 40),
                                      (4_096, 63, 40), (4_096, 64, 40), (4_096, 100, 40), (70_000, 100, 16),
                                      (4_096, 126, 40)])
@pytest.mark.parametrize("cut", [False, True])
def test_rows_on_the_conditions(oracle, v, k, rows, cut):
    from xwen_amd import sampler as xsm
    rng = np.random.default_rng(1000 * k + v + cut)
    ctx = xsm.Context(max_rows=rows, vocab=v)
    ctx.bind_current_stream()

    def sent():
        n = ctypes.c_uint32(0)
        assert ctx.lib.xs_test_serial_fallback(ctx.h, 0, ctypes.byref(n)) == 0
        return int(n.value)
    X, A, U, P, want, must = [], [], [], [], [], []
    weak = near = order_only = 0
    made = [_row(rng, v, k, [0.25, 1.0, 4.0][r % 3]) for r in range(rows)]
    T = [1.0, 0.7, 1.3][k % 3]
    xs = np.stack([m[0] for m in made])
    masked = np.where(np.stack([m[1] for m in made]), xs, -np.inf).astype(np.float32)
    # the device's exact sums: the same values without a mask, which no check applies to
    d = run_sample(ctx, masked, T, 2, 0.5, 0.5, enc=v, stats=True)
    assert (d["status"] == 0).all()
    for r, (x, allow, at) in enumerate(made):
        S = np.float32(d["soft_sum"][r])
        inv = np.float32(1.0 / T)
        s = (masked[r] * inv).astype(np.float32) if T != 1.0 else masked[r]
        order = np.lexsort((np.arange(v), -masked[r]))[:k + 2]
        e = np.array([oracle.exp(float(s[i] - s.max())) for i in order], np.float32)
        p = np.sort((e[:k] / S).astype(np.float32))[::-1]
        w, top_p, renorm = p, 1.0, cut
        if cut:
            sumc = np.float32(-0.0)
            for t in p:
                sumc = np.float32(sumc + t)
            w = (p / sumc).astype(np.float32)
        c = _chain(w)
        if cut:  # on a prefix sum, an ulp or two beside it, or a margin's width away
            j = int(rng.integers(0, k - 1))
            g = float(c[j]) * (1.0 + float(rng.choice([0, 1, -1, 2, k // 2 + 3, -k // 2 - 3])) * 2.0 ** -24)
            top_p = float(np.float32(min(g, 1.0 - 2.0 ** -24)))
        keep, found = k, False
        if cut:
            for j in range(k):
                if c[j] >= np.float32(top_p):
                    keep, found = j + 1, True
                    break
        tot = c[keep - 1]
        pairs = [i + t for i in at for t in (0, 1) if i < k - 2 and 0 < i + t < keep - 1]
        if pairs and rng.random() < 0.5:  # well inside one of a pair's entries
            j = pairs[int(rng.integers(0, len(pairs)))]
            u = np.float32((float(c[j - 1]) + float(c[j])) / (2.0 * float(tot)))
        elif keep > 1 and rng.random() < 0.85:  # around a boundary
            j = int(rng.integers(0, keep - 1))
            off = int(rng.choice([0, 1, -1])) if rng.random() < 0.3 else int(rng.integers(-5 * k, 5 * k))
            u = np.float32(min(max(float(c[j]) / float(tot) + off * 2.0 ** -24, 0.0), 1 - 2.0 ** -24))
        else:
            u = np.float32(rng.random())
        xd = np.float32(u * tot)
        idx = sum(1 for j in range(k - 1) if (c[j] if j < keep - 1 else tot) <= xd)
        ids = [int(i) for i in order[:k + 1]]
        low = float(e[k + 1])
        # the finalizer bounds what lies below the selection by the next float,
        # and looks for the row's next value only where e ties across the edge
        just = np.nextafter(masked[r][order[k]], np.float32(-np.inf))
        just = float(oracle.exp(float((np.float32(just * inv) if T != 1.0 else just) - s.max())))
        verdicts, plains, drawn = set(), set(), set()
        for below in {low, just} if e[k - 1] == e[k] else {just}:
            fails, plain, amb = _order(e[:k + 1], ids, k, float(S), v, below)
            for f in (0.99, 1.01):  # f32 margins: a few roundings, far inside 1 %
                pl = _plain(c, u, idx, keep, k, found, renorm, float(S), top_p, f)
                rf = pl or _refined(c, w, u, idx, keep, k, found, renorm, float(S), top_p, f)
                verdicts.add(fails or not rf or idx in amb)
                plains.add(plain and pl)
                drawn.add(not fails and rf)
        if len(verdicts) > 1:
            near += 1  # within 1 % of a margin, or the two bounds below the selection differ
        must.append(verdicts.pop() if len(verdicts) == 1 else None)
        weak += must[-1] is False and plains == {False}
        order_only += must[-1] is True and drawn == {True}  # (the drawn entry lies in a run)
        ctl = oracle.Ctl(allowed=workloads.pack_mask(allow[None, :])[0])
        want.append(oracle.sample_controlled(x, v, T, k, top_p, u=float(u), sum_mode=oracle.SUM_SEQ_F32,
                                             ctl=ctl).token)
        X.append(x)
        A.append(allow)
        U.append(u)
        P.append(top_p)
    X, U, P, mask = np.stack(X), np.array(U, np.float32), np.array(P), workloads.pack_mask(np.stack(A))
    before, got = sent(), []
    for r in range(rows):  # one row a call: which of them went to the serial sum
        n0 = sent()
        d = run_sample(ctx, X[r:r + 1], T, k, P[r:r + 1], U[r:r + 1], enc=v, mask=mask[r:r + 1], cand_k=0,
                       stats=False)
        got.append(sent() - n0)
        assert d["status"][0] == 0
        assert d["token"][0] == want[r], (r, int(d["token"][0]), want[r], got[r], must[r])
        assert must[r] is None or got[r] == int(must[r]), (r, got[r], must[r], float(U[r]), float(P[r]))
    total = sent() - before
    d = run_sample(ctx, X, T, k, P, U, enc=v, mask=mask, cand_k=0, stats=False)  # and all of them in one
    assert d["token"].tolist() == want and sent() - before == 2 * total
    print(f"\nv {v} k {k} cut {cut}: {total} of {rows} rows summed serially, {weak} settled by the weaker "
          f"conditions, {order_only} sent by the drawn entry's run alone, {near} too close to call")
    assert total >= 1 and weak >= 1 and near <= rows // 2 and (rows < 40 or order_only >= 1)
    ctx.close()
