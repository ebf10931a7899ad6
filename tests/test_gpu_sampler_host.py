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
