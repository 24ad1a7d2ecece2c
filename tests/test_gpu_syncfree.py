"""Sync-free triangular sweeps (one launch per sweep or
pair of sweeps; rows drawn in topological order; the output pre-filled with a
sentinel that marks unfinished rows; each row's dependency values staged
through LDS behind a bounded, wave-voted wait; strips of rows for narrow levels)
against the CPU oracle, and against the level-scheduled sweeps."""

import numpy as np
import pytest

from conftest import rel
from helpers import heat, seepage

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fctx(B):
    c = B.Context()
    c.set_sweep_mode(1)
    return c


def dev(B, x):
    return B.DeviceArray.from_host(np.asfortranarray(x))


@pytest.mark.parametrize("nrhs", [1, 2, 5, 6])
def test_syncfree_ic2_sweeps(B, O, fctx, nrhs):
    h = heat(B, O, 9, 8, 9, seed=5)
    U = h["U"]
    print(f"syncfree ic2 nrhs={nrhs} nsup={U.nsup}", flush=True)
    x = np.random.default_rng(3).standard_normal((U.n, nrhs))
    dx, dy, dz = dev(B, x), B.DeviceArray((U.n, nrhs)), B.DeviceArray((U.n, nrhs))
    fctx.solve_l(h["f"], 1, dx, dy, nrhs)
    fctx.solve_u(h["f"], 1, dy, dz, nrhs)
    fctx.sync()
    y = O.solvel(U, x, nrhs)
    assert rel(dy.host(), y) < 1e-13
    assert rel(dz.host(), O.solveu(U, y, nrhs)) < 1e-13


def test_syncfree_ilu2_all_directions(B, O, fctx):
    s = seepage(B, O, 6, 5, 4, 24, seed=6)
    L, U = s["L"], s["U"]
    print(f"syncfree ilu2 nsup={L.nsup}", flush=True)
    x = np.random.default_rng(4).standard_normal(L.n)
    dx, dy = dev(B, x), B.DeviceArray(L.n)
    for which, fn, ref in ((0, fctx.solve_l, O.solvel(L, x)), (1, fctx.solve_l, O.solvel(U, x)),
                           (1, fctx.solve_u, O.solveu(U, x)), (0, fctx.solve_u, O.solveu(L, x))):
        fn(s["f"], which, dx, dy)
        fctx.sync()
        assert rel(dy.host(), ref) < 1e-13


@pytest.mark.parametrize("precision,tol", [(1, 2e-5), (2, 2e-2)])
def test_syncfree_low_precision(B, O, fctx, precision, tol):
    s = seepage(B, O, 5, 4, 3, 24, seed=7)
    r = np.random.default_rng(5).standard_normal(s["A"].n)
    ref = O.solveu(s["U"], O.solvel(s["L"], r))
    dr, dz = dev(B, r), B.DeviceArray(s["A"].n)
    fctx.precond(s["f"], dr, dz, precision=precision)
    fctx.sync()
    assert rel(dz.host(), ref) < tol


def test_syncfree_solvers(B, O, fctx):
    h = heat(B, O, 16, 14, 9, seed=11)
    db, dx = dev(B, h["b"]), B.DeviceArray(h["A"].n)
    dx.zero()
    st = fctx.solve(h["mo"], h["f"], db, dx, B.default_opts(kind=B.PCG, eps=1e-10, ittype=0))
    xo, r = O.cg(h["A"], h["U"], h["b"], eps=1e-10, ittype=0)
    assert st.converged and st.iterations == r.updates and rel(dx.host(), xo) < 1e-8
    s = seepage(B, O, 6, 5, 4, 24, seed=12)
    db, dx = dev(B, s["b"]), B.DeviceArray(s["A"].n)
    dx.zero()
    st = fctx.solve(s["mo"], s["f"], db, dx, B.default_opts(kind=B.BICGSTAB, eps=1e-10))
    xo, r = O.bicgstab(s["A"], s["L"], s["U"], s["b"], eps=1e-10)
    assert st.converged and st.relres_true <= 1e-10 and rel(dx.host(), xo) < 1e-8


def coupled_groups(B, size, ngroup, blocks, seed):
    """Groups of `size` block rows, every row coupled to every other of its
    group: `size` dependency levels of `ngroup` rows, up to size - 1 blocks a
    row. `blocks` lists the block sizes, row after row (repeated)."""
    rng = np.random.default_rng(seed)
    ns = size * ngroup
    bs = np.array([blocks[k % len(blocks)] for k in range(ns)])
    vals, ja = [], []
    for r in range(ns):
        for c in range(r // size * size, r // size * size + size):
            blk = 0.2 * rng.standard_normal((bs[c], bs[r]))
            if c == r:
                blk = blk + 8.0 * np.eye(bs[r])
            vals.append(blk.ravel())
            ja.append(c)
    sp = np.concatenate([[0], np.cumsum(bs)]).astype(np.int32)
    m = B.Matrix.from_arrays(sp, np.arange(ns + 1) * size, ja, np.concatenate(vals), False)
    return m, B.Factor.ilu2(m, B.default_params(tau1=1e-9, tau2=1e-11))


# 600 groups of 3: levels of 600 rows, 16 rows a workgroup (blocks up to 16) or
# three columns a wave and a rest of one (above: 400 x 7); 16 columns of 400
# rows: by levels above 16; 12 groups of 9: narrow levels, one wave per column,
# and rows of 8 dependencies (more than the chunks held in registers)
GROUPS = [(3, 600, 2), (3, 600, 3), (3, 400, 7), (3, 400, 16), (9, 12, 1), (9, 12, 6), (9, 200, 6)]


@pytest.mark.parametrize("size,ngroup,nrhs", GROUPS)
@pytest.mark.parametrize("b", [3, 6, 8, 9, 12, 16, 24, 32])
def test_syncfree_pair_matches_level_schedule(B, fctx, b, size, ngroup, nrhs):
    if b > 16 and size * ngroup * size > 6000:
        size, ngroup = 3, 400  # bounded host factorization
    m, f = coupled_groups(B, size, ngroup, [b], seed=b)
    print(f"pair b={b} groups {ngroup} x {size} nrhs={nrhs}", flush=True)
    r = np.random.default_rng(6).standard_normal((m.n, nrhs))
    lctx = B.Context()
    lctx.set_sweep_mode(0)
    # the same products per row in another order: sums of up to 9 * 32 terms, FP32 factors and vectors for precision 1 and 2
    for precision, tol in ((0, 1e-13), (1, 2e-5), (2, 2e-5)):
        dr, dz, dl = dev(B, r), B.DeviceArray((m.n, nrhs)), B.DeviceArray((m.n, nrhs))
        fctx.precond(f, dr, dz, nrhs, precision=precision)
        lctx.precond(f, dr, dl, nrhs, precision=precision)
        fctx.sync()
        lctx.sync()
        want = dl.host()
        assert rel(dz.host(), want) < tol
        fctx.precond(f, dr, dr, nrhs, precision=precision)  # in place
        fctx.sync()
        assert rel(dr.host(), want) < tol


def complex_precond(ns, b, low, up, x):
    """(U D)^-1-type application in numpy, row by row: low by columns, up by
    rows, inverted diagonal blocks first, blocks column-major."""
    (lia, lja, la), (uia, uja, ua) = low, up
    v = x.reshape(ns, b, -1).copy()
    lb, ub = la.reshape(-1, b, b), ua.reshape(-1, b, b)  # transposed blocks
    for i in range(ns):
        v[i] = lb[lia[i]] @ v[i]
        for j in range(lia[i] + 1, lia[i + 1]):
            v[lja[j]] -= lb[j] @ v[i]
    y = v.copy()
    for i in range(ns - 1, -1, -1):
        for j in range(uia[i] + 1, uia[i + 1]):
            v[i] -= ub[j].T @ v[uja[j]]
        v[i] = ub[uia[i]].T @ v[i]
    return y.reshape(x.shape), v.reshape(x.shape)


# 400 groups of 3: wide levels; 30 groups of 8: rows with more dependencies than
# two chunks hold. Against complex arithmetic in numpy, in every schedule.
@pytest.mark.parametrize("bc,size,ngroup,nrhs", [(3, 3, 400, 2), (12, 3, 400, 3), (16, 3, 400, 6), (4, 3, 400, 6), (3, 8, 30, 1),
                                                 (4, 8, 30, 2), (6, 8, 30, 7), (8, 8, 30, 1), (12, 9, 20, 1), (16, 8, 12, 2)])
def test_syncfree_complex_levels(B, fctx, bc, size, ngroup, nrhs):
    rng = np.random.default_rng(8)
    ns = size * ngroup
    ia, ja = [0], []
    for r in range(ns):
        ja += list(range(r, r // size * size + size))
        ia.append(len(ja))
    ia, ja = np.array(ia), np.array(ja)
    sp = np.arange(ns + 1) * bc
    low, up = [(ia, ja, (0.1 * (rng.standard_normal((len(ja), bc, bc)) + 1j * rng.standard_normal((len(ja), bc, bc)))).ravel())
               for _ in range(2)]
    f = B.Factor.from_complex(sp, low, up)
    print(f"complex levels bc={bc} groups {ngroup} x {size} nrhs={nrhs}", flush=True)
    z = rng.standard_normal((ns * bc, nrhs)) + 1j * rng.standard_normal((ns * bc, nrhs))
    y, want = complex_precond(ns, bc, low, up, z)
    dr = dev(B, B.complex_to_real(sp, z))
    dz, dn = B.DeviceArray((2 * ns * bc, nrhs)), B.DeviceArray((2 * ns * bc, nrhs))
    try:
        for mode in (1, 2, 0):
            fctx.set_sweep_mode(mode)
            fctx.solve_l(f, 0, dr, dz, nrhs)
            fctx.sync()
            assert rel_c(B.real_to_complex(sp, dz.host()), y) < 1e-13, mode
            fctx.precond(f, dr, dz, nrhs)
            fctx.precond_noalloc(f, dr, dn, nrhs)
            fctx.sync()
            assert rel_c(B.real_to_complex(sp, dz.host()), want) < 1e-12, mode
            assert np.array_equal(dz.host(), dn.host()), mode
    finally:
        fctx.set_sweep_mode(1)


def rel_c(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


# Any block partition: one-row blocks, the largest (64), and rows whose
# dependencies span more columns than are staged at a time (8 x 64 > 192).
@pytest.mark.parametrize("blocks,size,ngroup,nrhs", [
    ([1], 3, 40, 1), ([64, 1, 33], 9, 6, 2), ([5, 7, 14, 11], 4, 50, 1), ([10], 9, 20, 3), ([64], 5, 4, 6)])
def test_syncfree_any_partition_matches_level_schedule(B, fctx, blocks, size, ngroup, nrhs):
    m, f = coupled_groups(B, size, ngroup, blocks, seed=3)
    print(f"any partition {blocks} groups {ngroup} x {size} nrhs={nrhs}", flush=True)
    r = np.random.default_rng(7).standard_normal((m.n, nrhs))
    lctx = B.Context()
    lctx.set_sweep_mode(0)
    for precision, tol in ((0, 1e-13), (1, 2e-5), (2, 2e-5)):
        for transpose in (False, True):
            dr, dz, dl = dev(B, r), B.DeviceArray((m.n, nrhs)), B.DeviceArray((m.n, nrhs))
            fctx.precond(f, dr, dz, nrhs, precision=precision, transpose=transpose)
            lctx.precond(f, dr, dl, nrhs, precision=precision, transpose=transpose)
            fctx.sync()
            lctx.sync()
            assert rel(dz.host(), dl.host()) < tol
        dy, dm = B.DeviceArray((m.n, nrhs)), B.DeviceArray((m.n, nrhs))
        if precision == 0:
            for fn in ("solve_l", "solve_u"):
                getattr(fctx, fn)(f, 1, dr, dy, nrhs)
                getattr(lctx, fn)(f, 1, dr, dm, nrhs)
                fctx.sync()
                lctx.sync()
                assert rel(dy.host(), dm.host()) < 1e-13


# Chains of coupled groups: as many levels as rows.
@pytest.mark.parametrize("b,size,ngroup,nrhs", [
    (3, 4, 8, 1), (6, 4, 60, 2), (8, 5, 83, 1), (9, 4, 90, 6), (12, 4, 70, 1), (16, 3, 50, 3), (16, 4, 12, 1)])
def test_syncfree_strips_match_level_schedule(B, fctx, b, size, ngroup, nrhs):
    rng = np.random.default_rng(b)
    ns = size * ngroup  # a chain of coupled groups: row r depends on the rest of its group and the group before
    ia, ja, vals = [0], [], []
    for r in range(ns):
        k = r // size * size
        cols = list(range(max(0, k - (size if r == k else 0)), k + size))
        if r == k + size - 1 and k + size < ns:
            cols.append(k + size)
        for c in cols:
            blk = 0.1 * rng.standard_normal((b, b))
            ja.append(c)
            vals.append((blk + 8.0 * np.eye(b) if c == r else blk).ravel())
        ia.append(len(ja))
    m = B.Matrix.from_arrays(np.arange(ns + 1) * b, ia, ja, np.concatenate(vals), False)
    f = B.Factor.ilu2(m, B.default_params(tau1=1e-6, tau2=1e-8))
    print(f"strips b={b} ns={ns} nrhs={nrhs}", flush=True)
    r = rng.standard_normal((m.n, nrhs))
    lctx = B.Context()
    lctx.set_sweep_mode(0)
    for precision, tol in ((0, 1e-13), (1, 2e-5), (2, 2e-5)):
        for transpose in (False, True):
            dr, dz, dl = dev(B, r), B.DeviceArray((m.n, nrhs)), B.DeviceArray((m.n, nrhs))
            fctx.precond(f, dr, dz, nrhs, precision=precision, transpose=transpose)
            lctx.precond(f, dr, dl, nrhs, precision=precision, transpose=transpose)
            fctx.sync()
            lctx.sync()
            assert rel(dz.host(), dl.host()) < tol


def grid_system(B, nx, ny, b, seed):
    """An nx x ny grid, small couplings on a large diagonal: the factor keeps the
    pattern. Every tenth row of a line has seven more earlier neighbours, of its
    own strip and of others; no row is one of more than one such row. Levels stay
    the antidiagonals of the grid."""
    rng = np.random.default_rng(seed)
    i, j = np.divmod(np.arange(nx * ny), nx)
    pairs = []
    for di, dj in ((0, 1), (1, 0), (0, 2), (0, 3), (1, 1), (2, 0), (3, 4), (1, 5), (5, 6)):
        keep = (i >= di) & (j >= dj) & ((di + dj == 1) | (j % 10 == 9))
        r = np.flatnonzero(keep)
        pairs.append(np.stack([r, r - di * nx - dj], axis=1))
    lo = np.concatenate(pairs)
    ns = nx * ny
    r = np.concatenate([lo[:, 0], lo[:, 1], np.arange(ns)])
    c = np.concatenate([lo[:, 1], lo[:, 0], np.arange(ns)])
    o = np.lexsort((c, r))
    r, c = r[o], c[o]
    a = rng.standard_normal((len(r), b, b)) / b
    a[r == c] += 1000.0 * np.eye(b)
    ia = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=ns))])
    m = B.Matrix.from_arrays(np.arange(ns + 1) * b, ia, c, a.ravel(), False)
    return m, B.Factor.ilu2(m, B.default_params(tau1=1e-5, tau2=1e-5))


# Strips: every block size they are built for; rows with more dependencies than
# are held (nine: the leading five or six in two chunks), several rows of a level
# in a strip, strips of three and more rows a wave, columns.
@pytest.mark.parametrize("b,nx,ny,nrhs", [(3, 10, 103, 1), (6, 11, 372, 2), (8, 12, 341, 1), (9, 20, 660, 1), (9, 41, 40, 6),
                                          (12, 13, 485, 1), (16, 13, 485, 1), (16, 33, 30, 2)])
def test_syncfree_strips_with_leading_dependencies(B, plan, fctx, b, nx, ny, nrhs):
    m, f = grid_system(B, nx, ny, b, seed=b)
    for bytes_ in (8, 4, 2):
        strips, deps, shared = plan.factor_strips(f, nx * ny, b, bytes_, nrhs)
        assert strips and deps == 9 and (shared or nx > 20)
    print(f"strips b={b} grid {nx} x {ny} nrhs={nrhs}", flush=True)
    r = np.random.default_rng(6).standard_normal((m.n, nrhs))
    lctx = B.Context()
    lctx.set_sweep_mode(0)
    # couplings are some 1e-4 of the diagonal: a wrong or missing one shows far above the tolerances
    for precision, tol in ((0, 1e-13), (1, 2e-5), (2, 2e-5)):
        for transpose in (False, True):
            dr, dz, dl = dev(B, r), B.DeviceArray((m.n, nrhs)), B.DeviceArray((m.n, nrhs))
            for _ in range(2):
                fctx.precond(f, dr, dz, nrhs, precision=precision, transpose=transpose)
            lctx.precond(f, dr, dl, nrhs, precision=precision, transpose=transpose)
            fctx.sync()
            lctx.sync()
            assert rel(dz.host(), dl.host()) < tol


def test_syncfree_more_positions_than_a_launch(B, fctx):
    """70000 rows x 512 columns x 2 sweeps are 71.7 million waves, more than the
    2^32 threads that one launch takes."""
    ns, nrhs = 70000, 512
    m, f = coupled_groups(B, 2, ns // 2, [1], seed=4)
    print(f"{ns} rows x {nrhs} columns", flush=True)
    r = np.asfortranarray(np.random.default_rng(8).standard_normal((ns, nrhs)))
    lctx = B.Context()
    lctx.set_sweep_mode(0)
    dr, dz, dl = dev(B, r), B.DeviceArray((ns, nrhs)), B.DeviceArray((ns, nrhs))
    fctx.precond(f, dr, dz, nrhs)
    lctx.precond(f, dr, dl, nrhs)
    fctx.sync()
    lctx.sync()
    assert rel(dz.host(), dl.host()) < 1e-13


def chain(B, ns, b, seed):
    """Block-tridiagonal system and its ILU2 factor, which is then exact: one
    row a level, as many levels as rows."""
    rng = np.random.default_rng(seed)
    rows = np.arange(ns)
    ja = np.stack([rows - 1, rows, rows + 1], axis=1)
    keep = (ja >= 0) & (ja < ns)
    a = 0.2 * rng.standard_normal((ns, 3, b, b))
    a[:, 1] += 4.0 * np.eye(b)
    ia = np.concatenate([[0], np.cumsum(keep.sum(axis=1))])
    m = B.Matrix.from_arrays(np.arange(ns + 1) * b, ia, ja[keep], a[keep].ravel(), False)
    return m, a  # a[r, j]: transposed block (r, r - 1 + j)


@pytest.mark.parametrize("ns,b", [(1000000, 3), (60000, 16)])
def test_syncfree_long_chain(B, fctx, ns, b):
    """A million levels: rows wait for as long as the sweep lasts, with no
    other reason to give up (0.4 s a sweep, most of it polls of values within
    a strip). M = A here, so M^-1 (A x) = x."""
    m, a = chain(B, ns, b, seed=b)
    f = B.Factor.ilu2(m, B.default_params(tau1=1e-9, tau2=1e-11))
    print(f"long chain ns={ns} b={b}", flush=True)
    x = np.random.default_rng(9).standard_normal((ns, b))
    ax = np.einsum("rcb,rc->rb", a[:, 1], x)
    ax[1:] += np.einsum("rcb,rc->rb", a[1:, 0], x[:-1])
    ax[:-1] += np.einsum("rcb,rc->rb", a[:-1, 2], x[1:])
    dr, dz = dev(B, ax.ravel()), B.DeviceArray(m.n)
    fctx.precond(f, dr, dz)
    fctx.sync()
    # dominant diagonal blocks: nothing grows along the chain, and ILU2 drops what is below 1e-9
    assert rel(dz.host(), x.ravel()) < 1e-7
    y = dz.host()
    fctx.precond(f, dr, dz)
    fctx.sync()
    assert np.array_equal(dz.host(), y)
