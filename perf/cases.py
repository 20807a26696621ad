"""The work that a user of libssq has it do, as timed cases.

Every case is one call of a public entry point, or one batch through the server.  The inputs are
the workloads that this repository's configurations, tests and benchmark use: Vietoris-Rips
complexes of point clouds (uniform cube, noisy circle, noisy torus, rotations), thresholded at
the 30th distance percentile or at a mean vertex degree, and alpha complexes of uniform points.

Entries:
  points    Handle.batch_reduce_points: clouds from the host, pairs to the host
  stream    Handle.batch_reduce_points_device: points in HBM, pairs left in HBM
  reduce    Handle.reduce: one Rips matrix from the host (homology, cohomology, the models)
  alpha     Handle.reduce_device: one alpha matrix in HBM, pairs left in HBM
  resident  Handle.batch_reduce_resident: alpha matrices kept in HBM
  batch     Handle.batch_reduce: Rips matrices from the host as one batch
  build     Handle.vr_build_gpu: the Rips boundary matrix alone
  serve     Server: clouds and registered alpha matrices submitted together, all results polled

The seed moves the points, so the numbers of cells and pairs change a little with it.  Every
output goes to the front of a buffer that the program keeps, whose size follows from the case.
"""
import functools
import math
from types import SimpleNamespace

import numpy as np
import torch

import specseqplusplus_amd as S
from specseqplusplus_amd import configs, workloads
from specseqplusplus_amd.alpha import alpha_complex
from specseqplusplus_amd.server import Server

SHAPES = ("cube", "circle", "torus")
# parameters of the batched stream and of the served requests, as the benchmark sets them
STREAM = dict(dualize=1, ss_block_size=1 << 30, queue_size=16384, level1=64, level2=1024)
ALPHA = dict(model=0, queue_size=20000, level1=1000, level2=16000)


def _case(name, entry, n, **kw):
    c = dict(name=name, entry=entry, shape="mixed", count=1, nmin=n, nmax=n, degree=0.0, maxdim=2, model=0, dualize=0)
    c.update(kw)
    return c


def listed():
    return [
        # one small cloud from the host: the smallest request, where launches and round trips count
        _case("points_one_small", "points", 96, shape="torus"),
        # one large sparse cloud, the largest request that a server takes
        _case("points_one_large", "points", 4000, shape="circle", degree=20.0),
        # a server's batch of clouds
        _case("points_served_batch", "points", 4096, nmin=64, count=24, degree=20.0),
        # one dense cloud with its points in HBM, near the largest of the batched stream
        _case("stream_one_dense", "stream", 1700, shape="torus"),
        # a slice of the batched stream
        _case("stream_many", "stream", 2048, nmin=64, count=40),
        # a plain small Rips matrix, homology (the reference's own use)
        _case("reduce_homology", "reduce", 512, shape="cube", degree=23.0),
        # one mid-size Rips matrix in cohomology (the anti-transpose, then the reduction)
        _case("reduce_cohomology", "reduce", 777, shape="torus", degree=110.0, dualize=1),
        # a large Rips matrix with edge collapse and guided clearing (model 3)
        _case("reduce_collapsed", "reduce", 4096, shape="rotations", degree=80.0, model=3),
        # a 3-dimensional Rips matrix with guided clearing (model 1)
        _case("reduce_cleared_dim3", "reduce", 300, shape="cube", degree=40.0, maxdim=3, model=1),
        # a large alpha matrix in HBM
        _case("alpha_large", "alpha", 60000, shape="cube", maxdim=3),
        # a server's batch of alpha matrices kept in HBM
        _case("alpha_resident_batch", "resident", 8000, nmin=350, shape="cube", count=16, maxdim=3),
        # clouds and registered matrices submitted to the server together
        _case("serve_mixed", "serve", 1500, nmin=64, count=24, degree=20.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    entry = rng.choice(["points", "points", "stream", "stream", "reduce", "reduce", "alpha", "resident", "batch", "build"])
    shape = rng.choice(SHAPES)
    name = ""
    if entry == "points":
        if rng.random() < 0.5:
            c = _case(name, entry, _log(rng, 40, 400), shape=shape)
        else:
            lo, hi = sorted((_log(rng, 30, 4096), _log(rng, 30, 4096)))
            c = _case(name, entry, hi, nmin=lo, count=_log(rng, 1, 31), degree=20.0)
    elif entry == "stream":
        if rng.random() < 0.5:
            c = _case(name, entry, _log(rng, 64, 1600), shape=shape)
        else:
            lo, hi = sorted((_log(rng, 64, 1000), _log(rng, 64, 1000)))
            c = _case(name, entry, hi, nmin=lo, count=_log(rng, 2, 40))
    elif entry == "reduce":
        kind = rng.randrange(4)
        if kind == 0:
            c = _case(name, entry, _log(rng, 60, 1200), shape=shape, degree=rng.uniform(8.0, 30.0))
        elif kind == 1:
            c = _case(name, entry, _log(rng, 150, 1000), shape=shape, degree=rng.uniform(20.0, 110.0), dualize=1)
        elif kind == 2:
            c = _case(name, entry, _log(rng, 500, 3500), shape="rotations", degree=rng.uniform(40.0, 80.0),
                      model=rng.choice([2, 3]), dualize=rng.choice([0, 1]))
        else:
            c = _case(name, entry, _log(rng, 60, 300), shape=shape, degree=rng.uniform(10.0, 40.0), maxdim=3, model=1)
    elif entry == "alpha":
        c = _case(name, entry, _log(rng, 400, 40000), shape="cube", maxdim=3, dualize=rng.choice([0, 0, 1]))
    elif entry == "resident":
        lo, hi = sorted((_log(rng, 350, 8000), _log(rng, 350, 8000)))
        c = _case(name, entry, hi, nmin=lo, shape="cube", count=_log(rng, 1, 16), maxdim=3)
    elif entry == "batch":
        lo, hi = sorted((_log(rng, 40, 300), _log(rng, 40, 300)))
        c = _case(name, entry, hi, nmin=lo, count=_log(rng, 2, 24), degree=rng.uniform(10.0, 30.0), dualize=rng.choice([0, 1]))
    else:
        c = _case(name, entry, _log(rng, 100, 3000), shape=shape, degree=rng.uniform(10.0, 60.0))
    del c["name"]
    return c


# ---- inputs ---------------------------------------------------------------------------------
def _sizes(case):
    """`count` point counts spread over [nmin, nmax] by their logarithm."""
    k, lo, hi = case["count"], case["nmin"], case["nmax"]
    if k == 1:
        return [hi]
    return [int(round(lo * (hi / lo) ** (i / (k - 1)))) for i in range(k)]


def _clouds(case, seed):
    """[(float32 points, threshold)]: the shapes in turn where the case mixes them."""
    rng = np.random.default_rng(seed)
    out = []
    for i, n in enumerate(_sizes(case)):
        if case["shape"] == "rotations":
            X = configs.haar_rotations(n, int(rng.integers(1 << 30)))
        else:
            kind = i % 3 if case["shape"] == "mixed" else SHAPES.index(case["shape"])
            X = workloads.make_cloud(rng, kind, n).astype(np.float32)
        q = 30.0 if case["degree"] == 0 else min(30.0, 100.0 * case["degree"] / max(n - 1, 1))
        out.append((X, workloads.percentile_threshold(X, q)))
    return out


def _alphas(case, seed):
    """Alpha complexes of uniform points, at the density of 1e5 points in a cube of side 100."""
    rng = np.random.default_rng(seed)
    return [alpha_complex(rng.random((n, 3)) * 100.0 * (n / 1e5) ** (1 / 3), 90.0) for n in _sizes(case)]


@functools.lru_cache(maxsize=1)
def _handle():
    """The engine handle that a program keeps for all its calls."""
    return S.Handle(0)


@functools.lru_cache(maxsize=1)
def _server():
    """The server that a program keeps, with the benchmark's settings."""
    return Server(streams=4, max_batch=32, max_batch_cells=4 << 20, p=S.params(**ALPHA), points_p=S.params(**STREAM))


def _serve_alphas(case):
    return dict(case, nmin=350, nmax=6000, count=max(1, case["count"] // 3))


class _DeviceMatrices:
    """Matrices resident in HBM, freed with the state."""

    def __init__(self, h, mats):
        self.h, self.dms = h, [h.to_device(m) for m in mats]

    def __del__(self):
        for dm in self.dms:
            self.h.free_device_matrix(dm)


class _Registered:
    """Matrices registered with the server, given back with the state."""

    def __init__(self, srv, mats):
        self.srv, self.ids = srv, [srv.register_matrix(m) for m in mats]

    def __del__(self):
        for i in self.ids:
            self.srv.unregister_matrix(i)


def _cells(case, n):
    """Upper bounds of one complex's edges and cells, for the buffers of its results."""
    if case["entry"] in ("alpha", "resident"):
        return 9 * n + 64, 31 * n + 512
    v, e, t, q = _rips_cells(n, case["degree"], case["maxdim"])
    e = min(1.02 * e + 64, n * (n - 1) / 2)  # the threshold is a percentile of the distances
    return int(e), int(v + e + 6 * t + 20 * q + 512)


class _Kept:
    """Results side by side in one buffer: each its pairs and essential cells at the front of its
    own stretch, -1 behind them."""

    def __init__(self, room):
        self.base = np.concatenate([[0], np.cumsum(room)]).astype(np.int64)
        self.buf = np.full(int(self.base[-1]), -1, np.int64)

    def put(self, results):
        for b, (pairs, essential) in zip(self.base, results):
            k = 2 * len(pairs)
            self.buf[b:b + k] = pairs.reshape(-1)
            self.buf[b + k:b + k + len(essential)] = essential
        return self.buf


def _room(case):
    return [_cells(case, n)[1] for n in _sizes(case)]


def _params(case):
    if case["entry"] in ("points", "stream"):
        return S.params(**STREAM)
    if case["entry"] in ("alpha", "resident"):
        return S.params(**dict(ALPHA, dualize=case["dualize"]))
    kw = configs.C2_PARAMS if case["model"] >= 2 else configs.C1_PARAMS
    return S.params(**dict(kw, model=case["model"], dualize=case["dualize"]))


def prepare(case, seed):
    entry = case["entry"]
    s = SimpleNamespace(entry=entry, maxdim=case["maxdim"], p=_params(case))
    if entry in ("alpha", "resident"):
        mats = _alphas(case, seed)
    else:
        clouds = _clouds(case, seed)
    if entry == "serve":
        s.srv = _server()
        alphas = _alphas(_serve_alphas(case), seed + 1)
        s.registered = _Registered(s.srv, alphas)
        s.clouds = clouds
        s.kept = _Kept(_room(case) + [_cells(dict(entry="alpha"), n)[1] for n in _sizes(_serve_alphas(case))])
        return s
    s.h = _handle()
    if entry not in ("stream", "alpha", "build"):
        s.kept = _Kept(_room(case))
    if entry in ("points", "build"):
        s.clouds = clouds
        if entry == "build":
            e, n = _cells(case, case["nmax"])
            s.kept = np.full(n + 1, -1, np.int64), np.full(4 * n, -1, np.int32), np.full(n, -1, np.int32)
    elif entry == "stream":
        s.pbase = np.concatenate([[0], np.cumsum([len(X) for X, _ in clouds])]).astype(np.int64)
        s.radius = np.array([r for _, r in clouds], np.float32)
        s.points = torch.from_numpy(np.concatenate([X for X, _ in clouds])).cuda()
        s.cap = sum(n + _cells(case, n)[0] for n in _sizes(case))  # one pair per vertex and edge
        s.pairs = torch.full((2 * s.cap,), -1, dtype=torch.int64, device="cuda")
    elif entry in ("reduce", "batch"):
        s.mats = [S.vr_build(X, r, case["maxdim"]) for X, r in clouds]
    elif entry == "alpha":
        m, = mats
        s.n, s.nnz = m.n, m.nnz
        s.matrix = [torch.from_numpy(a).cuda() for a in (m.colptr, m.rows, m.dims)]
        s.pairs = torch.full((2 * _cells(case, case["nmax"])[1],), -1, dtype=torch.int64, device="cuda")
    else:
        s.resident = _DeviceMatrices(s.h, mats)
    return s


def run(s):
    if s.entry == "points":
        return s.kept.put(s.h.batch_reduce_points(s.clouds, s.maxdim, s.p))
    if s.entry == "stream":
        off = s.h.batch_reduce_points_device(SimpleNamespace(ptr=s.points.data_ptr()), s.pbase, s.radius,
                                             SimpleNamespace(ptr=s.pairs.data_ptr()), s.cap, s.p)
        return s.pairs, off
    if s.entry == "reduce":
        return s.kept.put([s.h.reduce(s.mats[0], s.p)])
    if s.entry == "alpha":
        colptr, rows, dims = (t.data_ptr() for t in s.matrix)
        count, _ = s.h.reduce_device(s.n, s.nnz, colptr, rows, dims, s.pairs.data_ptr(), s.p)
        return s.pairs, count
    if s.entry == "resident":
        return s.kept.put(s.h.batch_reduce_resident(s.resident.dms, s.p))
    if s.entry == "batch":
        return s.kept.put(s.h.batch_reduce(s.mats, s.p))
    if s.entry == "build":
        (X, r), = s.clouds
        m = s.h.vr_build_gpu(X, r, s.maxdim)
        for k, a in zip(s.kept, (m.colptr, m.rows, m.dims)):
            k[:len(a)] = a
        return s.kept
    tickets = [s.srv.submit_points(X, r, s.maxdim) for X, r in s.clouds]
    tickets += [s.srv.submit_registered(i) for i in s.registered.ids]
    s.srv.wait_all()
    return s.kept.put([s.srv.poll(t)[:2] for t in tickets])


# ---- what a pass cannot do without -------------------------------------------------------------
def _rips_cells(n, degree, maxdim):
    """Expected edges and larger cliques of n points with a mean vertex degree: in a ball of a
    3-dimensional space 15/32 of the pairs of neighbours are neighbours, and about 0.27 of the
    triples all are."""
    d = degree if degree else 0.3 * (n - 1)
    e, t = n * d / 2, n * d * d / 6 * 0.47
    return n, e, t, (n * d ** 3 / 24 * 0.13 if maxdim >= 3 else 0.0)


def work(case):
    """Bytes of the inputs and outputs; operations: the distances (a subtraction, a product and a
    sum per coordinate) and one comparison per cell and facet of the complexes."""
    sizes, entry = _sizes(case), case["entry"]
    nbytes = flops = 0.0
    for n in sizes:
        if entry in ("alpha", "resident"):
            cells, nnz = 28.5 * n, 81.5 * n
        else:
            v, e, t, q = _rips_cells(n, case["degree"], case["maxdim"])
            cells, nnz = v + e + t + q, 2 * e + 3 * t + 4 * q
        matrix = 8 * (cells + 1) + 4 * nnz + 4 * cells
        if entry in ("points", "stream", "serve"):
            # the pairs are at most the edges; to the host every other cell comes back too
            nbytes += 12 * n + 16 * e + (0 if entry == "stream" else 8 * max(0.0, cells - 2 * e))
        elif entry == "build":
            nbytes += 12 * n + matrix
        else:
            nbytes += matrix + 8 * cells
        flops += nnz + (0 if entry in ("alpha", "resident") else 1.5 * 3 * n * n)
    return {"bytes": nbytes, "flops": flops}


# ---- the values, by a plain textbook reduction --------------------------------------------------
def _plain_rips(X, r, maxdim):
    """Cells of the Rips complex in (longest edge, dimension, vertices) order: (dims, facets)."""
    P = np.asarray(X, np.float64)
    acc = np.zeros((len(P), len(P)))
    for k in range(P.shape[1]):
        acc += (P[:, None, k] - P[None, :, k]) ** 2
    D = np.sqrt(acc).astype(np.float32)
    near = D <= np.float32(r)
    np.fill_diagonal(near, False)
    later = [set(np.flatnonzero(near[i, i + 1:]) + i + 1) for i in range(len(P))]
    cells = [(0.0, 0, (i,)) for i in range(len(P))]

    def grow(f, verts, cand):
        for v in sorted(cand):
            g = max([f] + [float(D[u, v]) for u in verts])
            cells.append((g, len(verts), verts + (v,)))
            if len(verts) < maxdim:
                grow(g, verts + (v,), cand & later[v])

    for i in range(len(P)):
        if maxdim > 0:
            grow(0.0, (i,), later[i])
    cells.sort()
    at = {c[2]: k for k, c in enumerate(cells)}
    facets = [sorted(at[c[2][:j] + c[2][j + 1:]] for j in range(len(c[2]))) if c[1] else [] for c in cells]
    return np.array([c[1] for c in cells], np.int32), facets


def _plain_pairs(dims, facets):
    """Column by column from the highest dimension down, columns as bit sets of rows."""
    pivot, death = {}, {}
    for d in range(int(dims.max()), 0, -1):
        for c in np.flatnonzero(dims == d):
            if c in death:  # the birth of a pair: it reduces to zero
                continue
            col = 0
            for f in facets[c]:
                col ^= 1 << f
            while col:
                low = col.bit_length() - 1
                if low not in pivot:
                    pivot[low] = col
                    death[low] = int(c)
                    break
                col ^= pivot[low]
    pairs = np.array(sorted(death.items()), np.int64).reshape(-1, 2)
    alone = np.ones(len(dims), bool)
    alone[pairs.reshape(-1)] = False
    return pairs, np.flatnonzero(alone).astype(np.int64)


def exact(case, seed):
    """Pairs, essential cells and matrices are whole numbers.  They are given for the small Rips
    complexes; an alpha complex would need another triangulation, and edge collapse changes the
    complex."""
    sizes, entry = _sizes(case), case["entry"]
    cells = sum(sum(_rips_cells(n, case["degree"], case["maxdim"])) for n in sizes)
    if entry in ("alpha", "resident", "serve") or case["model"] >= 2 or cells > 40000:
        return None
    plain = [_plain_rips(X, r, case["maxdim"]) for X, r in _clouds(case, seed)]
    if entry == "build":
        (dims, facets), = plain
        e, n = _cells(case, case["nmax"])
        kept = np.full(n + 1, -1, np.int64), np.full(4 * n, -1, np.int32), np.full(n, -1, np.int32)
        colptr = np.concatenate([[0], np.cumsum([len(f) for f in facets])])
        for k, a in zip(kept, (colptr, [f for col in facets for f in col], dims)):
            k[:len(a)] = a
        return kept
    found = [_plain_pairs(*m) for m in plain]
    if entry == "stream":
        off = np.concatenate([[0], np.cumsum([len(p) for p, _ in found])]).astype(np.int64)
        pairs = torch.full((2 * sum(n + _cells(case, n)[0] for n in sizes),), -1, dtype=torch.int64)
        pairs[:2 * int(off[-1])] = torch.from_numpy(np.concatenate([p for p, _ in found]).reshape(-1))
        return pairs, off
    return _Kept(_room(case)).put(found)
