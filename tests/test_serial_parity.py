"""The walk's shortcut for a segment with one half-way term (one_tie in
xs_sampler.hip), restated and checked against the serial f32 sum: such a
segment adds its grid units, the half-way term rounded down, and one unit more
when the sum before it plus the units through that term is odd.

The kernel's own sums are held bit for bit to the oracle's by the GPU tests of
the serial denominator; this pins the arithmetic, at every binade offset, with
the half-way term at every place of a short segment."""
import numpy as np
import pytest


def _units(e, grid):
    q = float(e) / grid
    fl = np.floor(q)
    fr = q - fl
    return int(fl) + (1 if fr > 0.5 else 0), fr == 0.5


@pytest.mark.parametrize("exponent", [-20, -3, 0, 5])
def test_one_half_way_term(exponent):
    rng = np.random.default_rng(exponent + 50)
    grid = 2.0 ** (exponent - 23)
    seen = 0
    for _ in range(400):
        n = int(rng.integers(1, 24))
        place = int(rng.integers(0, n))
        terms = [np.float32(grid * (float(rng.integers(0, 1 << 12)) + float(rng.integers(1, 1 << 9)) / 1024.0))
                 for _ in range(n)]  # fractions of 1/1024: never half-way
        terms[place] = np.float32(grid * (float(rng.integers(0, 1 << 12)) + 0.5))
        s = np.float32(2.0 ** exponent * (1.0 + float(rng.integers(0, 1 << 21)) * 2.0 ** -23))
        m = int(s.view(np.uint32))
        u = [_units(t, grid) for t in terms]
        assert sum(t for _, t in u) == 1
        par = sum(x for x, _ in u[:place + 1]) & 1
        got = m + sum(x for x, _ in u) + ((m + par) & 1)
        if got >> 23 != m >> 23:  # a carry: the kernel adds the terms
            continue
        for t in terms:
            s = np.float32(s + t)
        assert int(s.view(np.uint32)) == got
        seen += 1
    assert seen > 200
