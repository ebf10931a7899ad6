"""The Python Sampler's host buffers: calls of different row counts, options
changed between calls, row errors, controls, another stream, and a result that
a later call does not change, against the oracle."""
import numpy as np
import pytest

from tests import workloads

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

V = 40_003


def _want(oracle, x, opts, u, ctl=None):
    octl = None
    if ctl is not None:
        octl = oracle.Ctl(allowed=None)
        octl.banned, octl.bias, octl.pull, octl.force = tuple(ctl.banned), tuple(ctl.bias), ctl.pull, ctl.force
    return [oracle.sample_controlled(x[r], V, opts.temperature, opts.top_k, opts.top_p, u=float(u[r]),
                                     sum_mode=oracle.SUM_F64, ctl=octl).token for r in range(x.shape[0])]


def test_calls_share_the_buffers(oracle):
    from xwen_amd import sampler as xsm
    rng = np.random.default_rng(5)
    opts = xsm.SamplerOptions.recommended(thinking=False)
    s = xsm.Sampler(opts, [0], V, max_rows=8)
    kept = []
    for n, (t, k, p) in [(8, (0.7, 20, 0.8)), (1, (0.7, 20, 0.8)), (5, (0.0, 20, 0.8)), (8, (1.3, 50, 0.95))]:
        opts.temperature, opts.top_k, opts.top_p = t, k, p
        x = rng.standard_normal((n, V)).astype(np.float32) * np.float32(3.0)
        u = workloads.uniforms(rng, n)
        got = s.sample(torch.as_tensor(x).cuda(), u)
        want = _want(oracle, x, opts, u)
        assert got.dtype == np.int64 and got.tolist() == want
        kept.append((got, want))
    for got, want in kept:  # later calls left them alone
        assert got.tolist() == want
    opts.temperature, opts.top_k, opts.top_p = 0.7, 20, 0.8
    x = rng.standard_normal((3, V)).astype(np.float32)
    u = workloads.uniforms(rng, 3)
    bad = x.copy()
    bad[1, 17] = np.nan
    with pytest.raises(xsm.SampleError) as err:
        s.sample(torch.as_tensor(bad).cuda(), u)
    assert err.value.status.tolist() == [0, 1, 0]
    with pytest.raises(ValueError):
        s.sample(torch.as_tensor(x).cuda(), u[:1])
    ctl = xsm.SampleControl(banned=[int(x[0].argmax())], bias=[(9, 4.0)], pull=(11, 0.5))
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        xd = torch.as_tensor(x).cuda()
        assert s.sample_controlled(xd, ctl, u).tolist() == _want(oracle, x, opts, u, ctl)
    assert s.sample(torch.as_tensor(x).cuda(), u).tolist() == _want(oracle, x, opts, u)
    assert err.value.status.tolist() == [0, 1, 0]


def test_greedy_takes_fewer_uniforms(oracle):
    """Greedy rows ignore their uniforms, so a short array is as good as a full
    one; a stochastic sampler refuses it, and both refuse an empty one."""
    from xwen_amd import sampler as xsm
    x = np.random.default_rng(6).standard_normal((4, V)).astype(np.float32)
    xd = torch.as_tensor(x).cuda()
    for opts in (xsm.SamplerOptions(temperature=0.0), xsm.SamplerOptions(temperature=0.7, top_k=1)):
        s = xsm.Sampler(opts, [0], V, max_rows=4)
        for u in ([0.5], np.zeros(3, np.float32), np.zeros(9, np.float32)):
            assert s.sample(xd, u).tolist() == x.argmax(1).tolist()
        with pytest.raises(ValueError):
            s.sample(xd, [])
    s = xsm.Sampler(xsm.SamplerOptions(temperature=0.7), [0], V, max_rows=4)
    with pytest.raises(ValueError):
        s.sample(xd, [0.5])


def test_a_call_left_in_an_exception_keeps_its_block(oracle, monkeypatch):
    """A call interrupted after its launch leaves kernels that still read its
    uniforms and write its tokens: the next call, on another stream and before
    them, must not share their block, and the block is given back once they
    have run."""
    from xwen_amd import sampler as xsm
    rng = np.random.default_rng(7)
    opts = xsm.SamplerOptions(temperature=0.9, top_k=20, top_p=0.95)
    s = xsm.Sampler(opts, [0], V, max_rows=4)
    x = rng.standard_normal((4, V)).astype(np.float32) * np.float32(2.0)
    xd = torch.as_tensor(x).cuda()
    u1, u2 = workloads.uniforms(rng, 4), workloads.uniforms(rng, 4)
    want1, want2 = _want(oracle, x, opts, u1), _want(oracle, x, opts, u2)
    assert s.sample(xd, u2).tolist() == want2  # (options packed, buffers taken once)
    torch.cuda.synchronize()
    launch = xsm.sample_batch
    first = {}

    def interrupted(*a, out, **kw):
        torch.cuda._sleep(50_000_000)  # the launch waits on its stream: 20 ms or more
        launch(*a, out=out, **kw)
        first.update(u=a[3], token=out.token)
        raise KeyboardInterrupt

    slow = torch.cuda.Stream()
    with torch.cuda.stream(slow):
        monkeypatch.setattr(xsm, "sample_batch", interrupted)
        with pytest.raises(KeyboardInterrupt):
            s.sample(xd, u1)
        monkeypatch.setattr(xsm, "sample_batch", launch)
        assert len(s._stuck) == 1 and s._bufs is None
    fast = torch.cuda.Stream()
    with torch.cuda.stream(fast):
        got = s.sample(xd, u2)
    assert got.tolist() == want2
    assert s._bufs["host"].data_ptr() != first["u"].data_ptr()
    assert first["u"].numpy().view(np.float32)[:4].tolist() == u1.tolist()  # still what that launch will read
    slow.synchronize()
    assert first["token"].numpy()[:4].tolist() == want1
    assert s.sample(xd, u2).tolist() == want2 and not s._stuck
    with pytest.raises(xsm._lib.XsError):  # a refused call (more rows than the context holds)
        s.sample(torch.zeros((5, V), device="cuda"), np.zeros(5, np.float32))
    for u, want in ((u1, want1), (u2, want2)):
        assert s.sample(xd, u).tolist() == want and not s._stuck


def test_options_per_row(oracle):
    """Options set to one value a row, on a Sampler of more rows, between calls
    with numbers: each row draws with its own."""
    from xwen_amd import sampler as xsm
    rng = np.random.default_rng(8)
    opts = xsm.SamplerOptions(temperature=0.7, top_k=20, top_p=0.9)
    s = xsm.Sampler(opts, [0], V, max_rows=8)
    x = rng.standard_normal((3, V)).astype(np.float32) * np.float32(2.0)
    xd, u = torch.as_tensor(x).cuda(), workloads.uniforms(rng, 3)
    T, K, P = np.array([0.0, 0.6, 1.3]), [20, 50, 5], np.array([0.9, 1.0, 0.5])
    for t, k, p in [(0.7, 20, 0.9), (T, 20, 0.9), (T, K, P), (1.0, 20, P), (T + 0.1, K, P), (0.7, 20, 0.9)]:
        opts.temperature, opts.top_k, opts.top_p = t, k, p
        tt, kk, pp = (np.broadcast_to(np.asarray(a), (3,)) for a in (t, k, p))
        want = [oracle.sample_controlled(x[r], V, float(tt[r]), int(kk[r]), float(pp[r]), u=float(u[r]),
                                         sum_mode=oracle.SUM_F64).token for r in range(3)]
        for _ in range(2):
            assert s.sample(xd, u).tolist() == want
