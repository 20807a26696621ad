"""Guided clearing: how many top cells it clears, against a plain reading of its rule, with neighbour
lists on both sides of 64 and 2048 entries (sorted in registers, in LDS, by one lane) and
iteration limits on both sides of the 8 neighbours taken side by side.  Whole numbers: equal."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.complexes import closure_matrix

import specseqplusplus_amd as S

pytestmark = pytest.mark.gpu


def first_hits(m):
    """Per cleared cell, at which neighbour (from 0) the rule first holds."""
    n = len(m.dims)
    top = int(m.dims.max())
    facets = [m.rows[m.colptr[c]:m.colptr[c + 1]] for c in range(n)]
    verts, rank = {}, {}
    for c in range(n):
        if m.dims[c] == 0:
            rank[c] = len(rank)
            verts[c] = (rank[c],)
    for d in range(1, top + 1):
        for c in np.flatnonzero(m.dims == d):
            verts[c] = tuple(sorted(set().union(*(verts[f] for f in facets[c]))))
    nb = [[] for _ in rank]
    for c in np.flatnonzero(m.dims == 1):
        a, b = verts[c]
        nb[a].append(b)
        nb[b].append(a)
    near = [set(x) for x in nb]
    col = {verts[c]: c for c in np.flatnonzero(m.dims == top)}
    hits = []
    for c in np.flatnonzero(m.dims == top):
        v = verts[c]
        best = min(v, key=lambda a: (len(nb[a]), a))
        for k, x in enumerate(sorted(nb[best], reverse=True)):
            if x in v or any(x not in near[a] for a in v):
                continue
            others = [tuple(sorted((set(v) - {a}) | {x})) for a in v]
            if all(col.get(f, n) < c for f in others):
                hits.append(k)
                break
    return np.array(hits)


@pytest.fixture(scope="module")
def complexes():
    rng = np.random.default_rng(3)
    ms = [S.vr_build(rng.random((24, 3)).astype(np.float32), 2.0, 3)]  # complete
    for leaves in (63, 64, 65, 2047, 2048, 2049):  # tetrahedra's surfaces at a hub
        sets = [(0, i, i + 1, i + 2) for i in range(1, leaves - 1, 3)] + [(0, leaves - 1, leaves, 1)]
        ms.append(closure_matrix([s[:k] + s[k + 1:] for s in sets for k in range(4)], shuffle_seed=leaves))
    return [(S.Matrix(m.colptr, m.rows, m.dims), first_hits(m), O.twist_pairs(m)) for m in ms]


@pytest.mark.parametrize("limit", [0, 1, 2, 7, 8, 9, 17, 1 << 30])
def test_cleared_cells(complexes, limit):
    h = S.Handle(0)
    for m, hits, pairs in complexes:
        *out, st = h.reduce(m, S.params(model=1, max_iteration=limit), stats=True)
        assert st["n_cleared_hd"] == int((hits < limit).sum())
        assert np.array_equal(out[0], pairs)
    h.close()
