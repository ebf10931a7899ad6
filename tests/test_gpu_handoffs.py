"""The rare paths on every hand-off.  Rows whose entries overflow the finalizer's
list or a wave's stage (allow-masks of a few ranges at a wide top_k) and rows
with pulls and lists of every length, in calls whose rows are finalized by a
workgroup on another XCD (few rows), on the same one (64 rows and more), by
finalize_kernel (more workgroups than fit the device), under a row order, and
in verify blocks.  Every row is controlled, so its token is the serial-f32
reference's (oracle SUM_SEQ_F32)."""
import numpy as np
import pytest

from tests import workloads
from tests.test_gpu_sampler import oracle_row, run_sample

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# (rows, vocabulary): few rows; the XCD-local hand-off; more workgroups than the
# device holds, 16 a row and 4
SHAPES = [(6, 64_003), (64, 64_003), (71, 64_003), (66, 248_320), (264, 64_003)]


def _ranges(rng, rows, v):
    """Two thirds of the rows allow a few ranges, the others a tenth of the ids."""
    allow = np.zeros((rows, v), bool)
    for r in range(rows):
        if r % 3 == 2:
            allow[r] = rng.random(v, dtype=np.float32) < 0.1
            continue
        for _ in range(4):
            width = max(v // 400, 160)
            s = int(rng.integers(0, v - width))
            allow[r, s:s + width] = True
    return allow


def _masked(rows, v):
    """Masked rows whose lists overflow; values tied in eighths on every fifth row."""
    rng = np.random.default_rng(rows * 7 + v)
    ld = (v + 3) // 4 * 4
    x = rng.standard_normal((rows, ld), dtype=np.float32) * np.float32(3.0)
    x[::5] = np.round(x[::5] * 8) / np.float32(8)
    x[:, v:] = 50.0
    mask = workloads.pack_mask(_ranges(rng, rows, v))
    T = np.resize([0.8, 1.0, 0.6], rows)
    K = np.resize([50, 100, 63, 126, 20, 64], rows)
    P = np.resize([0.9, 1.0, 0.95, 1.0], rows)
    return x, T, K, P, workloads.uniforms(rng, rows), mask, None


def _controlled(rows, v):
    """Lists of 1 to 600 entries, pulls (of listed, forced, largest ids) on half the rows."""
    from xwen_amd import sampler as xsm
    rng = np.random.default_rng(rows * 11 + v)
    ld = (v + 3) // 4 * 4
    x = rng.standard_normal((rows, ld), dtype=np.float32) * np.float32(3.0)
    x[:, v:] = 99.0
    ctls = []
    for r in range(rows):
        n = int(rng.choice([1, 3, 40, 300, 512, 513, 600]))
        ids = [int(i) for i in rng.integers(0, v, n)]
        top = int(x[r, :v].argmax())
        bias = [(i, float(np.float32(d))) for i, d in zip(ids[n // 2:], rng.normal(0, 3, n))]
        pull = None
        if r % 2:
            pull = (int([ids[0], ids[-1], top, rng.integers(0, v)][r // 2 % 4]), float(rng.choice([0.5, 1.0, 2.0])))
        force = int(pull[0]) if r % 13 == 7 and pull else None
        banned = [top] * (r % 3 == 0) + ids[:n // 2]
        ctls.append(xsm.SampleControl(banned=tuple(banned), bias=tuple(bias), pull=pull, force=force))
    T = np.resize([0.9, 1.0, 0.7], rows)
    K = np.resize([20, 50, 63, 100, 5], rows)
    P = np.resize([0.95, 1.0], rows)
    return x, T, K, P, workloads.uniforms(rng, rows), None, ctls


def _want(oracle, v, x, T, K, P, U, mask, ctls):
    out = []
    for r in range(x.shape[0]):
        o = oracle_row(oracle, x[r], v, T[r], K[r], P[r], U[r], None if mask is None else mask[r],
                       sum_mode=oracle.SUM_SEQ_F32, **({} if ctls is None else {"ctl": ctls[r]}))
        assert o.status == 0, (r, o.status)
        out.append(o.token)
    return out


@pytest.mark.parametrize("rows,v", SHAPES)
@pytest.mark.parametrize("rowset", [_masked, _controlled])
def test_rare_rows_in_a_batch(oracle, rows, v, rowset):
    from xwen_amd import sampler as xsm
    x, T, K, P, U, mask, ctls = rowset(rows, v)
    want = _want(oracle, v, x, T, K, P, U, mask, ctls)
    ctx = xsm.Context(max_rows=rows, vocab=v)
    ctx.bind_current_stream()
    lg, u = torch.as_tensor(x).cuda(), torch.as_tensor(U).cuda()
    p = xsm.params_tensor(T, K, P, rows, "cuda")
    m = None if mask is None else torch.as_tensor(mask.view(np.int32)).cuda()
    c = None if ctls is None else xsm.controls_tensor(ctls, "cuda")
    order = xsm.cost_order(T, K) if rows <= 256 else None
    for o in (None, order):  # (a second call finds the tickets as the first left them)
        d = xsm.sample_batch(ctx, lg, p, u, enc=v, allowed=m, controls=c, order=o)
        torch.cuda.synchronize()
        assert (d.status == 0).all()
        assert d.token.tolist() == want
    ctx.close()


@pytest.mark.parametrize("seqs,span,v", [(2, 5, 64_003), (16, 5, 64_003), (11, 6, 248_320)])
@pytest.mark.parametrize("rowset", [_masked, _controlled])
def test_rare_rows_in_a_verify_block(oracle, seqs, span, v, rowset):
    from xwen_amd import sampler as xsm
    rows = seqs * span
    x, T, K, P, U, mask, ctls = rowset(rows, v)
    want = _want(oracle, v, x, T, K, P, U, mask, ctls)
    rng = np.random.default_rng(seqs)
    drafts = np.array([[want[s * span + i] if (s + i) % 4 else int(rng.integers(0, v)) for i in range(span - 1)]
                       for s in range(seqs)], np.int32)
    ctx = xsm.Context(max_rows=rows, vocab=v)
    ctx.bind_current_stream()
    lg, u = torch.as_tensor(x).cuda(), torch.as_tensor(U).cuda()
    p = xsm.params_tensor(T, K, P, rows, "cuda")
    m = None if mask is None else torch.as_tensor(mask.view(np.int32)).cuda()
    c = None if ctls is None else xsm.controls_tensor(ctls, "cuda")
    for _ in range(2):
        vd = xsm.verify_batch(ctx, lg, seqs, span, p, u, torch.as_tensor(drafts).cuda(), enc=v, allowed=m, controls=c)
        torch.cuda.synchronize()
        for s in range(seqs):
            n = 0  # drafts accepted: the walk stops at the first row that draws something else
            while n < span - 1 and want[s * span + n] == drafts[s, n]:
                n += 1
            assert int(vd.accepted[s]) == n
            assert vd.committed[s, :n + 1].tolist() == want[s * span:s * span + n + 1]
    ctx.close()


def test_lists_of_every_candidate(oracle):
    """The rows' whole candidate lists at 64 rows and more."""
    from tests.test_gpu_sampler import check_rows
    from xwen_amd import sampler as xsm
    rows, v = 66, 64_003
    for rowset in (_masked, _controlled):
        x, T, K, P, U, mask, ctls = rowset(rows, v)
        ctx = xsm.Context(max_rows=rows, vocab=v)
        ctx.bind_current_stream()
        d = run_sample(ctx, x, T, K, P, U, enc=v, mask=mask, ctls=ctls, cand_k=128)
        assert (d["status"] == 0).all()
        check_rows(oracle, x, T, K, P, U, d, enc=v, mask=mask, margins=False, label=rowset.__name__, ctls=ctls)
        ctx.close()
