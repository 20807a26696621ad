"""Additions of short columns (k_add): pivots of a few rows added to columns of up to 1024 rows,
through the window of the column's top 64 rows and the overlay.  Graphs with a hub whose coboundary
column crosses the window (63-65, 130 rows) and the wavefront's LDS (1023-1030 rows), with random
edges and triangles whose chases fill the overlay, cancel equal tops and meet larger pivots.
Pairs are whole numbers: bit-exact against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.complexes import closure_matrix

import specseqplusplus_amd as S

pytestmark = pytest.mark.gpu


def hub_complex(leaves, seed):
    rng = np.random.default_rng(seed)
    top = [(0, i + 1) for i in range(leaves)]
    n = leaves + 1
    for _ in range(2 * leaves):
        a, b = rng.integers(1, n, 2)
        if a != b:
            top.append((a, b))
    for _ in range(leaves // 2):  # triangles, some with the hub
        t = set(rng.integers(0, n, 3).tolist())
        if len(t) == 3:
            top.append(tuple(t))
    return closure_matrix([tuple(int(x) for x in s) for s in top], shuffle_seed=seed)


@pytest.fixture(scope="module")
def h():
    hd = S.Handle(0)
    yield hd
    hd.close()


@pytest.mark.parametrize("leaves", [2, 31, 63, 64, 65, 130, 400, 1023, 1024, 1030])
def test_hub_columns(h, leaves):
    for seed in range(3):
        m = hub_complex(leaves, seed)
        ref = O.twist_pairs(m)
        mm = S.Matrix(m.colptr, m.rows, m.dims)
        for kw in ({"dualize": 1}, {"dualize": 0}, {"dualize": 1, "short_max": 64}, {"dualize": 1, "ss_block_size": 64}):
            assert np.array_equal(h.reduce(mm, S.params(**kw))[0], ref), (seed, kw)
