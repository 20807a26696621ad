"""The coboundary columns of the batched Rips builder (k_rc_side, k_rc_merge) where their staging
changes: clouds whose words of Q take one pass or several, columns with more foreign entries than
the LDS list holds or more entries than one piece of output, a vertex without neighbours, equal
lengths (lattices).  Whole numbers: bit-exact against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O

import specseqplusplus_amd as S

pytestmark = pytest.mark.gpu


def _cloud(kind, n):
    rng = np.random.default_rng(n)
    if kind == "dense":  # every pair an edge: n - 2 common neighbours
        return rng.random((n, 3)).astype(np.float32), 2.0
    if kind == "sparse":  # a few neighbours in many words, and a far point
        X = rng.random((n, 3)).astype(np.float32)
        X[-1] += 9
        return X, float((12.0 / n) ** (1 / 3) * 0.62)
    k = int(round(n ** 0.5))
    g = np.stack(np.meshgrid(np.arange(k), np.arange(k), [0], indexing="ij"), -1).reshape(-1, 3)
    return g.astype(np.float32), 2.9


@pytest.mark.parametrize("kind,sizes", [("dense", [1, 2, 3, 63, 64, 65, 129, 200]), ("sparse", [70, 1500, 4096]),
                                        ("lattice", [49, 400])])
def test_columns(kind, sizes):
    hd = S.Handle(0)
    try:
        clouds = [_cloud(kind, n) for n in sizes]
        outs = hd.batch_reduce_points(clouds, 2, S.params(dualize=1, ss_block_size=1 << 30))
        for (X, r), (pairs, ess) in zip(clouds, outs):
            m = S.vr_build(X, r, 2)
            assert np.array_equal(pairs, O.twist_pairs(O.Matrix(m.colptr, m.rows, m.dims))), len(X)
            assert 2 * len(pairs) + len(ess) == m.n
    finally:
        hd.close()


def test_long_columns():
    """A cloud of two tight clumps: columns of over 1024 foreign entries and 1100 entries in all."""
    rng = np.random.default_rng(5)
    n = 1160
    X = (rng.random((n, 3)) * 0.01).astype(np.float32)
    X[: n // 40] += 1.0
    hd = S.Handle(0)
    try:
        d_pts = hd.device_array(X)
        pb, rad = np.array([0, n]), np.array([0.02], np.float32)
        e, t = hd.rips_count(d_pts, pb, rad)
        d_pairs = hd.device_empty(2 * int(e[0] + n), np.int64)
        off = hd.batch_reduce_points_device(d_pts, pb, rad, d_pairs, int(e[0] + n))
        pairs = d_pairs.numpy(2 * int(off[-1])).reshape(-1, 2)
        # every triangle of a full simplex: H0 dies along n - 2 edges, every other edge in a triangle
        assert len(pairs) == n - 2 + (int(e[0]) - (n - 2))
        assert np.all(np.diff(pairs[:, 0]) > 0) and np.all(pairs[:, 0] < pairs[:, 1])
        assert len(np.unique(pairs)) == pairs.size and pairs.max() < n + int(e[0]) + int(t[0])
        a = hd.batch_reduce_points_device(d_pts, pb, rad, d_pairs, int(e[0] + n))
        assert np.array_equal(a, off) and np.array_equal(d_pairs.numpy(2 * int(off[-1])).reshape(-1, 2), pairs)
    finally:
        hd.close()
