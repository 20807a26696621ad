"""Host edge collapse of edge lists that are no simple graphs: two edges with the same ends (cells of a
general complex), loops, both; on both sides of the bit-set tables (16384 vertices).  The search for a
dominating vertex has to end, and the kept edges are pinned: they are those that trying every common
neighbour in turn gives.  The collapse runs in a process of its own under a time limit."""
import os
import subprocess
import sys
import zlib

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LISTS = 40


def edges(kind, big, seed):
    rng = np.random.default_rng(seed)
    n, m = int(rng.integers(2, 40)), int(rng.integers(1, 200))
    u, v = rng.integers(0, n, m), rng.integers(0, n, m)
    if kind == "double":
        u, v = u[u != v], v[u != v]
    if kind in ("loops", "simple"):
        P = np.array(list(dict.fromkeys((min(a, b), max(a, b)) for a, b in zip(u.tolist(), v.tolist())
                                        if kind == "loops" or a != b)), np.int32).reshape(-1, 2)
        u, v = P[:, 0], P[:, 1]
    if big:  # a star brings the vertices past the bit sets
        u, v = np.concatenate([u, np.zeros(17000)]), np.concatenate([v, 100 + np.arange(17000)])
    return u.astype(np.int32), v.astype(np.int32)


def kept_crc(kind, big, threads):
    import specseqplusplus_amd as S

    crc = 0
    for seed in range(LISTS if not big else LISTS // 4):
        u, v = edges(kind, big, seed)
        if len(u):
            crc = zlib.crc32(np.ascontiguousarray(S.collapse_edges(u, v, threads), np.uint8).tobytes(), crc)
    return crc


# crc32 of the kept edges of all lists
KEPT = {
    ("double", False): 3777774631,
    ("double", True): 3729100690,
    ("loops", False): 3652139030,
    ("loops", True): 1491173382,
    ("both", False): 1678009393,
    ("both", True): 1644871195,
}


@pytest.mark.parametrize("threads", [1, 4])
@pytest.mark.parametrize("kind, big", list(KEPT))
def test_ends_with_the_kept_edges(kind, big, threads):
    code = f"from tests.test_collapse_multigraph import kept_crc; print(kept_crc({kind!r}, {big}, {threads}))"
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    assert int(r.stdout) == KEPT[kind, big]


def test_simple_lists_are_the_oracles():
    """The same generator without loops and doubles, pinned by the oracle and not by numbers."""
    import specseqplusplus_amd as S
    from oracle import oracle as O

    for seed in range(LISTS):
        u, v = edges("simple", False, seed)
        if len(u):
            assert np.array_equal(S.collapse_edges(u, v, 2), O.collapse_edges(u, v)), seed
