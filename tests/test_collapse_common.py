"""Common neighbours in the host edge collapse, by the words of two bit-set rows and by the shorter
adjacency list: vertices of very different degrees, below, at and above the number of words, with either
end of an edge the shorter one.  Equal to the oracle's kept edges."""
import numpy as np
import pytest

from oracle import oracle as O

import specseqplusplus_amd as S


@pytest.mark.parametrize("n, m", [(3, 3), (64, 900), (129, 1500), (700, 9000), (2000, 6000), (2000, 20000)])
@pytest.mark.parametrize("threads", [1, 4])
def test_kept_edges_of_uneven_degrees(n, m, threads):
    rng = np.random.default_rng(n + m)
    u = rng.integers(0, n, m)
    v = (n * rng.random(m) ** 4).astype(np.int64)  # a few vertices are in most edges
    P = np.unique(np.column_stack([np.minimum(u, v), np.maximum(u, v)])[u != v], axis=0)
    P = P[rng.permutation(len(P))]
    flip = rng.random(len(P)) < 0.5
    a, b = np.where(flip, P[:, 1], P[:, 0]).astype(np.int32), np.where(flip, P[:, 0], P[:, 1]).astype(np.int32)
    assert np.array_equal(S.collapse_edges(a, b, threads), O.collapse_edges(a, b))
