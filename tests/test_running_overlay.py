"""Rows that come back above the top of a running column (k_add): while the low is an overlay row, a
pivot may put a window row back that had left the column at the top, and every row that left between
it and the former top then stands below the column's top.  The flush that follows has 64 lanes for
the overlay and all of those.

The matrices bring back the topmost of up to 63 cleared window rows.  Their cells are rows of dimension
0 and columns of dimension 1, so a column may hold any rows.  Each ends with the reduced column itself
and one small row toggled: its low is that row, and another one if a single row of the reduced column is
wrong.  The first test follows the wavefront's bookkeeping on the host and pins what the guard has to
hold; the GPU tests compare pairs with the oracle, bit by bit."""
import numpy as np
import pytest

from oracle import oracle as O

import specseqplusplus_amd as S

LANES = 64


class Overflow(Exception):
    pass


class Running:
    """The running column as k_add holds it: base, window of its top 64 rows, overlay."""

    def __init__(self, rows, below_low):
        self.base, self.overlay, self.peak = sorted(rows), set(), 0
        self.below_low = below_low  # the guard counts every dead window row below the low
        self.open()

    def open(self):
        self.top_at = len(self.base) - 1
        self.win = self.base[::-1][:LANES]
        self.alive = [True] * len(self.win)

    def dead(self, below):
        return [x for x, a in zip(self.win, self.alive) if not a and x < below]

    def top(self):
        return next((x for x, a in zip(self.win, self.alive) if a), -1)

    def lost(self):
        return self.dead(self.top())

    def flush(self):
        for x in self.lost():
            self.overlay ^= {x}
            if len(self.overlay) > LANES:
                raise Overflow
        gone = self.alive.index(True) if any(self.alive) else LANES
        self.base = sorted(set(self.base[:max(self.top_at + 1 - gone, 0)]) ^ self.overlay)
        self.overlay = set()

    def toggle(self, x):
        if x in self.win:
            k = self.win.index(x)
            self.alive[k] = not self.alive[k]
        else:
            self.overlay ^= {x}
            if len(self.overlay) > LANES:
                raise Overflow

    def add(self, pivot, low):
        out = self.dead(low) if self.below_low else self.lost()
        if len(self.overlay) + len(out) + len(pivot) > LANES:
            self.flush()
            self.open()
        for x in pivot:
            self.toggle(x)
        self.peak = max(self.peak, len(self.overlay) + len(self.lost()))

    def low(self):
        while True:
            while not any(self.alive) and self.top_at >= 0:
                self.base = self.base[:max(self.top_at + 1 - LANES, 0)]
                self.open()
            o, a = max(self.overlay, default=-1), self.top()
            if o != a or a < 0:
                return max(o, a)
            self.alive[self.alive.index(True)] = False
            self.overlay.discard(o)


def chase(column, pivots, below_low):
    """The column reduced by the pivots (each by its largest row), and the largest overlay needed."""
    q, by_low = Running(column, below_low), {max(p): p for p in pivots}
    low = max(column)
    while low in by_low:
        q.add(by_low[low], low)
        low = q.low()
    q.flush()
    return set(q.base), q.peak


def plain(column, pivots):
    col, by_low = set(column), {max(p): p for p in pivots}
    while col and max(col) in by_low:
        col ^= by_low[max(col)]
    return col


def returning(base_len, b_len, spread, seed):
    """Pivots of b_len rows that clear the base's top rows from above (each leaves a new low over them),
    and one that puts the topmost cleared row back."""
    rng = np.random.default_rng(seed)
    base = sorted(rng.choice(np.arange(200, 700), base_len - 1, replace=False).tolist())
    over = list(range(1000, 700, -1))  # lows above the base, falling
    top = over.pop(0)
    cleared = base[::-1][:min(62, base_len - 1) - int(rng.integers(0, 4))]  # one window row stays at least
    fresh = rng.permutation(np.arange(1, 200)).tolist()  # rows that no column holds
    column = set(base) | {top}
    pivots, todo, low = [], list(cleared), top
    while todo:
        nxt = over.pop(0)
        take, todo = todo[:max(b_len - 2 - spread, 1)], todo[max(b_len - 2 - spread, 1):]
        pivots.append({low, nxt} | set(take) | {fresh.pop() for _ in range(min(spread, len(fresh)))})
        low = nxt
    pivots.append({low, cleared[0]} | {fresh.pop() for _ in range(min(max(b_len - 2, 0), len(fresh)))})
    if seed % 2:  # and the chase goes on from the row that came back
        pivots.append({cleared[0], 0} | set(fresh[:1]))
    return column, pivots


def ranges_column():
    """The cleared rows 69-40 under lows 1000-994, then 69 back: 69 overlay lanes."""
    r = lambda a, b: set(range(a, b + 1))
    pivots = [{1000, 999, 998, 997} | r(500, 511), {999} | r(55, 69), {998} | r(40, 54),
              r(994, 997) | r(520, 531), {996} | r(540, 554), {995, 69}]
    return r(0, 69) | {1000}, pivots


def steps_column():
    """Five pivots of 16 rows: 56 cleared rows, the topmost back with the fifth."""
    R = [1000] + [600 - i for i in range(1, 64)]
    pivots = [{R[0], 950, *R[1:15]}, {950, 940, *R[15:29]}, {940, 930, *R[29:43]}, {930, 920, *R[43:57]},
              {920, R[1], *range(14)}]
    return set(R), pivots


CASES = {"ranges": ranges_column(), "steps": steps_column(), "steps_on": (steps_column()[0], steps_column()[1] + [{599, 200}])}
for _len in (63, 64, 65, 66, 128, 129, 200):
    for _b in (2, 3, 5, 6, 7, 8, 15, 16):
        CASES[f"len{_len}_rows{_b}"] = returning(_len, _b, (_len + _b) % 3 if _b > 5 else _b // 5, _len * 100 + _b)


def matrix(column, pivots):
    n = 1001
    reduced = plain(column, pivots)
    free = min(set(range(n)) - {max(p) for p in pivots} - reduced)  # no pivot's row
    cols = [sorted(p) for p in pivots] + [sorted(column), sorted(reduced ^ {free})]
    return O.Matrix.from_columns([[] for _ in range(n)] + cols, [0] * n + [1] * len(cols))


@pytest.mark.parametrize("name", CASES)
def test_guard_holds_on_the_host(name):
    column, pivots = CASES[name]
    assert max(map(len, pivots)) <= 16 and all(p for p in pivots)
    got, peak = chase(column, pivots, below_low=True)
    assert got == plain(column, pivots)
    assert peak <= LANES


def test_rows_below_the_top_alone_are_not_enough():
    """The guard that counts the rows below the top alive one only, on the same columns."""
    over = []
    for name, (column, pivots) in CASES.items():
        try:
            chase(column, pivots, below_low=False)
        except Overflow:
            over.append(name)
    assert {"ranges", "steps", "steps_on"} <= set(over) and len(over) > 10


def test_guard_holds_on_random_pivots():
    rng = np.random.default_rng(11)
    for _ in range(300):
        n = int(rng.integers(80, 400))
        pivots = []
        for low in rng.permutation(np.arange(1, n)).tolist()[:int(rng.integers(n // 2, n))]:
            lo = max(0, low - int(rng.integers(2, 120)))
            k = min(low - lo, int(rng.integers(0, 16)))
            pivots.append({low} | set(rng.choice(np.arange(lo, low), k, replace=False).tolist()))
        column = set(rng.choice(n, int(rng.integers(1, n)), replace=False).tolist())
        got, peak = chase(column, pivots, below_low=True)
        assert got == plain(column, pivots) and peak <= LANES


@pytest.fixture(scope="module")
def h():
    hd = S.Handle(0)
    yield hd
    hd.close()


@pytest.mark.gpu
@pytest.mark.parametrize("name", CASES)
def test_returning_rows(h, name):
    m = matrix(*CASES[name])
    ref = O.twist_pairs(m)
    mm = S.Matrix(m.colptr, m.rows, m.dims)
    for kw in ({"dualize": 0, "model": 0}, {"dualize": 1, "model": 0}, {"dualize": 0, "model": 0, "queue_size": 1}):
        assert np.array_equal(h.reduce(mm, S.params(**kw))[0], ref), kw


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["ranges", "steps", "len63_rows16", "len64_rows2", "len200_rows15"])
def test_bytes_of_a_chase(h, name):
    """add_bytes is 4(|a| + |b| + |a ^ b|) + 24 for each addition of the one chase (no row of these
    columns is in the overlay and in the base at once)."""
    column, pivots = CASES[name]
    cols = [sorted(p) for p in pivots] + [sorted(column)]
    m = O.Matrix.from_columns([[] for _ in range(1001)] + cols, [0] * 1001 + [1] * len(cols))
    st = h.reduce(S.Matrix(m.colptr, m.rows, m.dims), S.params(model=0, ss_block_size=1 << 30), stats=True)[-1]
    by_low, a, want, longest = {max(p): p for p in pivots}, set(column), 0, 0
    while a and max(a) in by_low:
        b = by_low[max(a)]
        want += 4 * (len(a) + len(b) + len(a ^ b)) + 24
        longest = max(longest, len(a) + len(b))
        a = a ^ b
    assert (st["n_additions"], st["add_bytes"], st["max_addition_len"]) == (len(pivots), want, longest)


@pytest.mark.gpu
def test_bytes_of_a_long_chase(h):
    """A chase whose entries pass 32 bits: 2.2 million pivots of two rows, a column of 1001."""
    steps, kept = 2_200_000, 1000
    n = kept + steps + 1
    chain = np.stack([np.arange(kept, n - 1), np.arange(kept + 1, n)], 1)[::-1]  # {low - 1, low}
    rows = np.concatenate([chain.ravel(), np.arange(kept), [n - 1]]).astype(np.int32)
    colptr = np.concatenate([np.zeros(n, np.int64), 2 * np.arange(steps + 1), [len(rows)]]).astype(np.int64)
    dims = np.concatenate([np.zeros(n), np.ones(steps + 1)]).astype(np.int32)
    pairs, _, st = h.reduce(S.Matrix(colptr, rows, dims), S.params(model=0, ss_block_size=1 << 30), stats=True)
    assert len(pairs) == steps + 1 and pairs[0].tolist() == [kept, n + steps]
    a = kept + 1
    assert (st["n_additions"], st["add_bytes"]) == (steps, steps * (4 * (2 * a + 2) + 24))
