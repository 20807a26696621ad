"""Pivots of one step shared by wavefronts (k_add_long, k_add_huge): one to nine apparent pivots near the low,
of lengths around what one, two, four and eight wavefronts take in one load, added to a column held as a
bit set, and single pivots that are not apparent.  The last column is the reduced one with row 0 added, which no
other column holds: its low is 0, and another row if one row of the reduced column is wrong.  Pairs are whole
numbers: bit-exact against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O

import specseqplusplus_amd as S

pytestmark = pytest.mark.gpu
LENGTHS = [1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1025, 4097]
BELOW = 6000  # rows below the lows


def step(count, length, seed):
    rng = np.random.default_rng(seed)
    lows = list(range(BELOW, BELOW + count))
    lower = lambda k: set((1 + rng.choice(BELOW - 1, k, replace=False)).tolist())
    pivots = [lower(length - 1) | {low} for low in lows]
    column = lower(1500) | set(lows)
    reduced = set(column)
    for p in pivots:
        reduced ^= p
    return pivots, [column, reduced ^ {0}]


def chain(count, length, seed):
    """Pivots that hold the next pivot's low: not apparent, one to a step."""
    rng = np.random.default_rng(seed)
    lower = lambda k: set((1 + rng.choice(BELOW - 1, k, replace=False)).tolist())
    pivots = [lower(max(length - 2, 0)) | {low, low - 1} for low in range(BELOW + count, BELOW, -1)]
    column = lower(1500) | {BELOW + count}
    reduced = set(column)
    for p in pivots:
        reduced ^= p
    return pivots, [column, reduced ^ {0}]


def matrix(pivots, columns):
    n = BELOW + 16
    cols = [sorted(c) for c in pivots + columns]
    return O.Matrix.from_columns([[] for _ in range(n)] + cols, [0] * n + [1] * len(cols))


@pytest.mark.parametrize("window", [None, 128, 4224])
@pytest.mark.parametrize("kind", [step, chain])
@pytest.mark.parametrize("count", [1, 2, 3, 4, 5, 7, 8, 9])
def test_steps_of_few_pivots(monkeypatch, kind, count, window):
    monkeypatch.setenv("SSQ_TEST_SHORT_MAX", "16")
    if window:
        monkeypatch.setenv("SSQ_TEST_WINDOW_BITS", str(window))
    h = S.Handle(0)
    try:
        for length in LENGTHS:
            m = matrix(*kind(count, length, 100 * count + length))
            got, _, st = h.reduce(S.Matrix(m.colptr, m.rows, m.dims), S.params(model=0), stats=True)
            assert np.array_equal(got, O.twist_pairs(m)), length
            assert st["n_dense_additions"] + st["n_huge_additions"] >= count
    finally:
        h.close()
