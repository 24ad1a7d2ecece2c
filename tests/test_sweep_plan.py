"""What the sync-free sweeps decide on the host from a factor's structure: the
strips, and how long a wait may last. No counterpart in the reference."""

import numpy as np
import pytest


def grid(nx, ny, extra, seed):
    """Dependency lists of a forward sweep over an nx x ny grid (left and upper
    neighbour); one row in `extra` (0: none) has up to seven more."""
    rng = np.random.default_rng(seed)
    ia, ja = [0], []
    for r in range(nx * ny):
        d = set()
        if r % nx:
            d.add(r - 1)
        if r >= nx:
            d.add(r - nx)
        if extra and r % extra == extra - 1 and r > 9:
            d |= set(int(v) for v in rng.integers(0, r, 7))
        ja += sorted(d)
        ia.append(len(ja))
    return np.array(ia, np.int32), np.array(ja, np.int32)


def mirrored(ia, ja):
    """The same lists with row r as row ns - 1 - r: a backward sweep."""
    ns = len(ia) - 1
    deps = [sorted(ns - 1 - c for c in ja[ia[r]:ia[r + 1]]) for r in range(ns - 1, -1, -1)]
    return (np.concatenate([[0], np.cumsum([len(d) for d in deps])]).astype(np.int32),
            np.array([c for d in deps for c in d], np.int32))


@pytest.mark.parametrize("forward", [True, False])
@pytest.mark.parametrize("b,nx,ny,extra", [(3, 8, 4, 0), (6, 1, 700, 0), (8, 61, 67, 10), (9, 120, 110, 10), (12, 33, 50, 9),
                                           (16, 40, 40, 10), (3, 3, 40000, 0)])
def test_strips_are_a_topological_cut(plan, b, nx, ny, extra, forward):
    ia, ja = grid(nx, ny, extra, seed=b)
    if not forward:
        ia, ja = mirrored(ia, ja)
    ns = nx * ny
    n, lev = plan.levels(ia, ja, forward)
    k, rows, ptr, code = plan.cut(b, 8, ia, ja, forward)
    assert k > 0 and ptr[0] == 0 and ptr[k] == ns and (np.diff(ptr) > 0).all()
    assert np.array_equal(np.sort(rows), np.arange(ns))
    assert np.diff(ptr).max() * b * 8 <= 48 << 10
    at = np.empty(ns, np.int64)
    at[rows] = np.arange(ns)
    strip = np.searchsorted(ptr, at, side="right") - 1
    for q in range(k):  # within a strip by level: no row waits for a later one of its own wave
        assert (np.diff(lev[rows[ptr[q]:ptr[q + 1]]]) >= 0).all()
    owner = np.repeat(np.arange(ns), np.diff(ia))
    assert (at[ja] < at[owner]).all()  # dependencies come first, in the same strip or an earlier one
    same = strip[ja] == strip[owner]
    assert np.array_equal(code[same], -1 - (at[ja[same]] - ptr[strip[ja[same]]]))
    assert np.array_equal(code[~same], ja[~same])
    if extra:
        assert np.diff(ia).max() > plan.l.held(b) and same.any() and (~same).any()


def test_no_strips_where_rows_or_levels_do_not_suit(plan):
    ia, ja = grid(40, 40, 4, seed=1)  # a quarter of the rows beyond what is held
    assert plan.cut(9, 8, ia, ja, True)[0] == 0
    ia, ja = np.arange(0, 1, dtype=np.int32), np.zeros(0, np.int32)
    assert plan.cut(9, 8, ia, ja, True)[0] == 0
    ia, ja = np.zeros(5001, np.int32), np.zeros(0, np.int32)  # one level of 5000 rows
    assert plan.cut(9, 8, ia, ja, True)[0] == 0
    ia, ja = grid(20, 20, 0, seed=1)
    assert plan.cut(24, 8, ia, ja, True)[0] == 0 and plan.cut(16, 8, ia, ja, True)[0] > 0


# rows, levels and columns as timed, with the winner
@pytest.mark.parametrize("b,bytes_,ns,levels,nrhs,strips", [
    (9, 8, 4096, 185, 1, 1), (9, 8, 4096, 185, 6, 1), (6, 8, 46656, 195, 1, 1), (6, 8, 46656, 195, 3, 0),
    (6, 8, 74088, 234, 1, 0), (3, 8, 490000, 2218, 1, 0), (3, 8, 1000000, 1000000, 1, 1), (12, 8, 27000, 90, 1, 1),
    (16, 8, 40000, 484, 1, 0), (16, 4, 40000, 484, 1, 1), (16, 8, 8000, 58, 3, 0), (16, 4, 8000, 58, 3, 1),
    (24, 8, 4096, 26, 1, 0), (9, 8, 31, 31, 1, 0), (9, 8, 32, 32, 1, 1)])
def test_strip_rule_on_both_sides_of_its_lines(plan, b, bytes_, ns, levels, nrhs, strips):
    assert plan.l.in_strips(b, bytes_, ns, levels, nrhs) == strips


def test_wait_bound_exceeds_any_sweep(plan):
    """At least five times what a sweep takes if every level costs 4 us, every
    further chunk of three dependencies 1 us and every block and column 2 ns."""
    rng = np.random.default_rng(2)
    for _ in range(2000):
        levels = int(10 ** rng.uniform(0, 9))
        deps = int(10 ** rng.uniform(0, 4))
        blocks = levels * deps
        nrhs = int(10 ** rng.uniform(0, 3))
        sweep = levels * (4e-6 + 1e-6 * (deps / 3)) + 2e-9 * blocks * nrhs
        assert plan.l.wait_seconds(levels, deps, blocks, nrhs) > 5 * sweep
    assert 4.0 < plan.l.wait_seconds(400, 8, 20000, 6) < 5.0  # an ordinary system: not for minutes
