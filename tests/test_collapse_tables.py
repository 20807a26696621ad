"""Host edge collapse on both sides of its bit-set table (16384 vertices): points on a curve with
noise, joined to their nearest neighbours, shortest edge first.  Equal to the oracle's kept edges."""
import numpy as np
import pytest

from oracle import oracle as O

import specseqplusplus_amd as S


@pytest.mark.parametrize("n", [2, 64, 65, 16384, 16385])
@pytest.mark.parametrize("threads", [1, 4])
def test_kept_edges(n, threads):
    rng = np.random.default_rng(n)
    p = np.column_stack([np.arange(n), rng.random(n) * 4, rng.random(n) * 4])
    u, v = [], []
    for k in range(1, min(n, 5)):
        u.append(np.arange(n - k))
        v.append(np.arange(k, n))
    u, v = np.concatenate(u), np.concatenate(v)
    order = np.argsort(((p[u] - p[v]) ** 2).sum(1), kind="stable")
    relabel = rng.permutation(n)
    u, v = relabel[u[order]].astype(np.int32), relabel[v[order]].astype(np.int32)
    lo, hi = np.minimum(u, v), np.maximum(u, v)
    assert np.array_equal(S.collapse_edges(lo, hi, threads), O.collapse_edges(lo, hi))
