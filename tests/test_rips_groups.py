"""Groups and streams of a batched Rips call (specseqplusplus_amd/csrc/ssq_groups.h), through the test
harness in tests/harness: every cloud in one group, groups within the budget and the cells, and no call
on fewer streams than it has groups and streams to run them on before a split."""
import ctypes
import os

import numpy as np
import pytest

HARNESS = os.path.join(os.path.dirname(os.path.abspath(__file__)), "harness", "libssq_groups_harness.so")
GROUP_CELLS, SPLIT_CELLS = 1 << 30, 1 << 23


def plan(sizes, budget, streams):
    if not os.path.exists(HARNESS):
        raise RuntimeError(f"{HARNESS} is not built; run __graft_entry__.build()")
    L = ctypes.CDLL(HARNESS)
    P, c64 = ctypes.c_void_p, ctypes.c_int64
    L.ssq_harness_groups.argtypes = [ctypes.c_int, P, P, P, c64, ctypes.c_int, P, P, P]
    a = np.array(sizes, np.int64).reshape(-1, 3)
    cols = [np.ascontiguousarray(a[:, k]) for k in range(3)]
    group, nbytes, workers = np.empty(len(a), np.int32), np.empty(len(a)), np.zeros(1, np.int32)
    assert L.ssq_harness_groups(len(a), *(c.ctypes.data for c in cols), budget, streams, group.ctypes.data,
                                nbytes.ctypes.data, workers.ctypes.data) == 0
    assert (group >= 0).all()
    return a.sum(1), group, nbytes, int(workers[0])


def cloud(n, degree=0):
    d = degree or 0.3 * (n - 1)
    return n, int(n * d / 2), int(n * d * d / 6 * 0.47)


def whole_groups(sizes, budget):
    """Groups before a split: on one stream a call is never split."""
    return plan(sizes, budget, 1)[1].max() + 1


@pytest.mark.parametrize("streams", [2, 3, 4, 8, 16])
@pytest.mark.parametrize("groups", [1, 2, 3, 4, 5, 7, 12, 15, 16, 20])
def test_no_fewer_streams_than_groups_before_a_split(groups, streams):
    sizes = [cloud(900)] * (4 * groups)
    one = plan(sizes, 1 << 60, 1)[2][0] - 64.0 * (1 << 20)
    budget = int(4.5 * one + 64.0 * (1 << 20))  # four clouds each
    assert whole_groups(sizes, budget) == groups
    cells, group, _, workers = plan(sizes, budget, streams)
    assert workers >= min(groups, streams)
    assert workers <= min(streams, group.max() + 1)


def test_no_fewer_streams_where_cells_make_the_groups():
    sizes = [cloud(2048)] * 60
    whole = whole_groups(sizes, 1 << 60)
    assert 4 <= whole < 16
    assert plan(sizes, 1 << 60, 16)[3] >= whole


@pytest.mark.parametrize("streams", [1, 2, 4, 16])
@pytest.mark.parametrize("budget", [1, 200_000_000, 9_000_000_000, 1 << 60])
def test_every_cloud_once_and_groups_within_bounds(budget, streams):
    rng = np.random.default_rng(streams)
    sizes = [cloud(int(n)) for n in np.exp(rng.uniform(np.log(3), np.log(2048), 50))] + [(0, 0, 0), (1, 0, 0)]
    cells, group, nbytes, workers = plan(sizes, budget, streams)
    order = np.argsort(-np.array(sizes)[:, 2], kind="stable")
    assert (np.diff(group[order]) >= 0).all()  # consecutive clouds by decreasing triangles
    for g in range(group.max() + 1):
        mine = group == g
        assert mine.any()
        assert mine.sum() == 1 or (cells[mine].sum() <= GROUP_CELLS and nbytes[mine].max() <= budget)
    assert 1 <= workers <= min(streams, group.max() + 1)


@pytest.mark.parametrize("total", [1_000_000, SPLIT_CELLS, 20_000_000, 200_000_000])
def test_a_call_in_one_group_is_split(total):
    sizes = [cloud(300)] * max(1, total // sum(cloud(300)))
    cells, group, _, workers = plan(sizes, 1 << 60, 4)
    assert plan(sizes, 1 << 60, 1)[1].max() == 0
    if cells.sum() <= SPLIT_CELLS:
        assert group.max() == 0 and workers == 1
    else:
        assert group.max() >= 1 and workers == min(3, group.max() + 1)
