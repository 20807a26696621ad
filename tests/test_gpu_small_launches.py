"""Sizes at which the engine goes from one workgroup to a grid: prefix sums of up to 16384 values
(one launch), and claim rounds over worklists of up to 2048 columns (claims and publishing in one
launch).  Whole numbers: equal to numpy's sums and to the oracle's pairs."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.complexes import closure_matrix
from tests.test_gpu_sort import harness, scan_on_gpu

import specseqplusplus_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 1023, 1024, 1025, 4097, 16383, 16384, 16385])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_scan_sizes(n, mode):
    x = np.random.default_rng(n).integers(0, 1000, n).astype([np.int32, np.uint32, np.int32][mode])
    want = np.cumsum(x.astype(np.int64))
    got = scan_on_gpu(harness(), x, mode)
    got = np.asarray(got)[:n + (mode != 2)]
    assert np.array_equal(got, want if mode == 2 else np.concatenate([[0], want]))


@pytest.mark.parametrize("block", [1, 1024, 2047, 2048, 2049, 6000])
@pytest.mark.parametrize("dualize", [0, 1])
def test_claim_rounds(block, dualize):
    rng = np.random.default_rng(block)
    e = rng.integers(0, 3000, (9000, 2))
    t = rng.integers(0, 3000, (3000, 3))
    top = [tuple(int(x) for x in s) for s in list(e) + list(t) if len(set(s.tolist())) == len(s)]
    m = closure_matrix(top, shuffle_seed=block)
    h = S.Handle(0)
    got = h.reduce(S.Matrix(m.colptr, m.rows, m.dims), S.params(dualize=dualize, ss_block_size=block))[0]
    h.close()
    assert np.array_equal(got, O.twist_pairs(m))


@pytest.mark.parametrize("sizes", [(900, 60), (900, 850, 64, 800, 3)])
def test_call_split_over_streams(monkeypatch, sizes):
    """A call of more than 8 million cells is split into groups on several streams: pairs as on one
    stream, where it is one group."""
    rng = np.random.default_rng(len(sizes))
    clouds = [(rng.random((n, 3)).astype(np.float32), 0.55) for n in sizes]
    results = []
    for streams in ("1", "4"):
        monkeypatch.setenv("SSQ_RIPS_STREAMS", streams)
        h = S.Handle(0)
        *out, st = h.batch_reduce_points(clouds, 2, S.params(dualize=1), stats=True)
        h.close()
        results.append((out[0] if len(out) == 1 else out, st["n_pages"]))
    (one, g1), (many, g4) = results
    assert g1 == 1 and g4 > 1
    for (a, ae), (b, be) in zip(one, many):
        assert np.array_equal(a, b) and np.array_equal(ae, be)
