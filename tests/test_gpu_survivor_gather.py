"""Rows whose published keys bound their selection weakly or not at all, so that
more entries pass the bound than the finalizer's list holds (256): small
vocabularies at wide top_k, allow-masks of a few ranges, values tied at the
bound, and values ascending by id (each entry read displaces an earlier one).
Token, candidates and weights against the CPU oracle, as every sampler row."""
import numpy as np
import pytest

from tests import workloads
from tests.test_gpu_sampler import check_held_row, check_rows, run_sample

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _uniforms(rng, n):
    return rng.integers(0, 1 << 23, n).astype(np.float32) * np.float32(2.0 ** -23)


@pytest.mark.parametrize("vocab,masked,shape", [
    (1_024, False, "ascending"),     # one chunk of one slot: 4 sub-records, all full
    (19_450, False, "normal"),       # two chunks: 32 published keys below K' = 101
    (19_450, False, "ties"),         # eighths: dozens of entries tied at the bound
    (32_771, False, "ascending"),    # 12 sub-records, a last slot of three ids
    (28_474, True, "normal"),        # a few allowed ranges, all of them kept
    (64_003, True, "ties"),
    (248_320, True, "normal"),       # 64 sub-records, four ranges of 620 ids
    (300_001, True, "normal"),       # more than 64 sub-records: nothing preloaded past them
])
def test_more_entries_than_the_list_holds(oracle, vocab, masked, shape):
    from xwen_amd import sampler as xsm
    rng = np.random.default_rng(vocab + masked)
    rows = 6
    ld = (vocab + 3) // 4 * 4
    x = (rng.standard_normal((rows, ld), dtype=np.float32) * np.float32(3.0))
    if shape == "ties":
        x = np.round(x * 8) / np.float32(8)
    elif shape == "ascending":
        x = np.sort(x, axis=1)
    x[:, vocab:] = 50.0  # past the encodable ids: never read
    mask = None
    if masked:
        allow = np.zeros((rows, vocab), bool)
        for r in range(rows):
            if r % 3 == 2:
                allow[r] = rng.random(vocab) < 0.1
                continue
            for _ in range(4):
                width = max(vocab // 400, 160)
                s = int(rng.integers(0, vocab - width))
                allow[r, s:s + width] = True
        mask = workloads.pack_mask(allow)
    T = np.array([0.8, 1.0, 0.6] * 2)
    K = np.array([50, 100, 63, 127, 20, 64])
    P = np.array([0.9, 1.0, 0.95] * 2)
    U = _uniforms(rng, rows)
    ctx = xsm.Context(max_rows=rows, vocab=vocab)
    ctx.bind_current_stream()
    d = run_sample(ctx, x, T, K, P, U, enc=vocab, mask=mask, cand_k=128)
    assert (d["status"] == 0).all(), d["status"]
    check_rows(oracle, x, T, K, P, U, d, enc=vocab, mask=mask, margins=False, label=f"{vocab} {shape}")
    if mask is None:  # the n_top highest logits come from the same selection
        d = run_sample(ctx, x, T, K, P, U, enc=vocab, cand_k=128, n_top=100)
        for r in range(rows):
            check_held_row(oracle, x[r, :vocab], d, r, 100, label=f"{vocab} {shape}")
    ctx.close()
