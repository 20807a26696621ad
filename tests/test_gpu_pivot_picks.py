"""Additions of several pivots per step (k_add_long, k_add_huge): noisy circles and lattices in
cohomology, whose chases add thousands of apparent pivots.  The LDS window and the device region
are made small enough that steps cross groups of four words, window moves, pivots that reach
below the window or the region, and lists that fill up.  Pairs are whole numbers: bit-exact
against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O

import specseqplusplus_amd as S
from specseqplusplus_amd import workloads as W

pytestmark = pytest.mark.gpu


def _clouds():
    rng = np.random.default_rng(11)
    out = [W.make_cloud(rng, 1, n).astype(np.float32) for n in (31, 127, 260)]
    out.append(W.make_cloud(rng, 2, 300).astype(np.float32))
    g = np.stack(np.meshgrid(np.arange(14), np.arange(14), [0], indexing="ij"), -1).reshape(-1, 3)
    out.append(g.astype(np.float32))  # equal lengths: blocks of rows shared by many columns
    return [(X, W.percentile_threshold(X, 30.0)) for X in out]


@pytest.mark.parametrize("window,region", [(None, None), (128, None), (128, 1 << 12), (128, 1 << 20),
                                           (4224, 1 << 16), (1 << 18, 1 << 18)])
def test_picked_pivots(window, region, monkeypatch):
    monkeypatch.setenv("SSQ_TEST_SHORT_MAX", "16")
    if window:
        monkeypatch.setenv("SSQ_TEST_WINDOW_BITS", str(window))
    if region:
        monkeypatch.setenv("SSQ_TEST_GLOBAL_BITS", str(region))
    hd = S.Handle(0)
    try:
        clouds = _clouds()
        outs, st = hd.batch_reduce_points(clouds, 2, S.params(dualize=1, ss_block_size=1 << 30), stats=True)
        assert st["n_dense_additions"] + st["n_huge_additions"] + st["n_tiled_additions"] > 1000
        for (X, r), (pairs, _) in zip(clouds, outs):
            m = S.vr_build(X, r, 2)
            assert np.array_equal(pairs, O.twist_pairs(O.Matrix(m.colptr, m.rows, m.dims))), len(X)
            for kw in ({"dualize": 1, "ss_block_size": 4096}, {"dualize": 0}):  # pages; homology
                assert np.array_equal(hd.reduce(m, S.params(**kw))[0], pairs), (len(X), kw)
    finally:
        hd.close()
