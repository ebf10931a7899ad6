"""control_kernel's chunk workgroups: a pulled row's max is taken by one
workgroup per chunk over its unlisted ids, and short lists are sorted by
counting.  Lists at the sort's edges (0, 1, 512, 513 entries), listed maxima in
first and last chunks, pulls whose target is listed, forced, masked or the
maximum itself, vocabularies that end inside a chunk, a slot and a float4.
Against the CPU oracle, and a second call on the same context (the tickets are
left zero)."""
import numpy as np
import pytest

from tests import workloads
from tests.test_gpu_sampler import check_rows, run_sample

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,masked", [(1_021, False), (16_384, True), (16_387, False), (40_001, True),
                                          (248_320, False), (300_001, True)])
def test_pulls_and_list_lengths(oracle, vocab, masked):
    from xwen_amd import sampler as xsm
    S = xsm.SampleControl
    rng = np.random.default_rng(vocab)
    rows = 10
    ld = (vocab + 3) // 4 * 4
    x = rng.standard_normal((rows, ld), dtype=np.float32) * np.float32(3.0)
    x[:, vocab:] = 99.0  # past the encodable ids: not part of the max
    x[1, vocab - 1] = 30.0  # the max in the last chunk, listed (below)
    x[2, 0] = 30.0          # in the first, not listed
    x[3, vocab - 1] = np.nan if not masked else 30.0
    mask = None
    if masked:
        allow = rng.random((rows, vocab)) < 0.5
        allow[3, vocab - 1] = False  # the max is masked out
        allow[:, 7] = True
        mask = workloads.pack_mask(allow)

    def ids(n):
        return [int(i) for i in rng.integers(0, vocab, n)]

    def bias(n):
        return tuple((i, float(np.float32(d))) for i, d in zip(ids(n), rng.normal(0, 3, n)))

    ctls = [S(pull=(7, 0.5)),                                             # no list
            S(banned=(vocab - 1,), pull=(7, 1.0)),                        # one entry: the max
            S(bias=((7, 1.5), (7, -0.25)), pull=(7, 2.0)),                # the target listed
            S(banned=tuple(ids(100)), bias=bias(412), pull=(7, 0.75)),    # 512 entries
            S(banned=tuple(ids(1)), bias=bias(512), pull=(7, 0.75)),      # 513
            S(banned=tuple(ids(300)), bias=bias(300)),                    # no pull
            S(pull=(7, 0.5), force=7),                                    # the forced id is the pulled one
            S(bias=bias(3), pull=(7, 0.5), force=9),
            S(bias=((11, 40.0),), pull=(11, 1.0)),                        # the target is the max
            None]
    T, K, P = np.full(rows, 0.9), np.array([20, 50, 5, 40, 63, 20, 20, 20, 100, 20]), np.full(rows, 0.95)
    U = (rng.integers(0, 1 << 23, rows) * 2.0 ** -23).astype(np.float32)
    ctx = xsm.Context(max_rows=rows, vocab=vocab)
    ctx.bind_current_stream()
    for _ in range(2):
        d = run_sample(ctx, x, T, K, P, U, enc=vocab, mask=mask, cand_k=128, ctls=ctls)
        check_rows(oracle, x, T, K, P, U, d, enc=vocab, mask=mask, margins=False, label=f"{vocab}", ctls=ctls)
    ctx.close()
