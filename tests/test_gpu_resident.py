"""The resident solves (lfgpu_resident.hip) against the two-sweep solver.

opts->graph = -1 runs the sweeps, 0 (the default) the resident solve where
the system fits the chip.  Both run the same recurrences and stop on the same
test with sums in another order.  Where the recurrence has lost
orthogonality (chains here take more iterations than they have rows) rounding
moves the count, so counts are compared over three iterations only.
Solutions: the
matrices here have no eigenvalue below 1e-3, so two converged solutions differ
by at most 2 rtol ||b|| / 1e-3 (a tenth more for the recurrence residual's
distance from the true one).
"""
import ctypes
import time

import numpy as np
import pytest

from lehrfempp_amd import capi

pytestmark = pytest.mark.gpu

MODES = [capi.PCG_FP64, capi.PCG_MIXED, capi.PCG_MIXED_MATRIX]


@pytest.fixture(scope="module")
def ctx():
    with capi.Context(0) as c:
        yield c


def _lattice_system(S, L, steps, seed, symmetric=True):
    """Triplets of a lattice Laplacian (S rows a line, L lines, neighbours
    (dx, dy) in steps and their opposites) with random weights plus 1e-3."""
    rng = np.random.default_rng(seed)
    n = S * L
    y, x = np.divmod(np.arange(n), S)
    rows, cols, vals, diag = [], [], [], np.full(n, 1e-3)
    for dx, dy in steps:
        i = np.nonzero((x + dx >= 0) & (x + dx < S) & (y + dy < L))[0]
        j = i + dy * S + dx
        w = np.exp(rng.standard_normal(i.size))
        rows += [i, j]
        cols += [j, i]
        vals += [-w, -w if symmetric else -w * (1.0 + 1e-15 * rng.integers(0, 2, i.size))]
        np.add.at(diag, i, w)
        np.add.at(diag, j, w)
    rows.append(np.arange(n))
    cols.append(np.arange(n))
    vals.append(diag)
    return np.concatenate(rows), np.concatenate(cols), np.concatenate(vals), n


def _flipped_system(S, L, seed):
    """_lattice_system with half of the squares cut along the other diagonal."""
    r, c, v, n = _lattice_system(S, L, ((1, 0), (0, 1), (1, 1)), seed)
    rng = np.random.default_rng(seed + 1)
    d = np.nonzero(c - r == S + 1)[0]
    d = d[rng.random(d.size) < 0.5]
    back = np.nonzero(r - c == S + 1)[0]
    pos = np.zeros(n, np.int64)
    pos[c[back]] = back  # the entry (i + S + 1, i) by i
    r2, c2 = r.copy(), c.copy()
    r2[d], c2[d] = r[d] + 1, c[d] - 1
    r2[pos[r[d]]], c2[pos[r[d]]] = c[d] - 1, r[d] + 1
    diag = np.full(n, 1e-3)  # (row sums move with the couplings)
    off = r2 != c2
    np.subtract.at(diag, r2[off], v[off])
    v2 = v.copy()
    v2[~off] = diag[r2[~off]]
    return r2, c2, v2, n


def _compare(ctx, A, n, mode, seed, x0=None, maxit=20000, rtol=1e-10):
    bh = np.random.default_rng(seed).standard_normal(n)
    b, bn = capi.Vec(ctx, bh), np.linalg.norm(bh)
    out = []
    for graph in (-1, 0):
        x = capi.Vec(ctx, np.zeros(n) if x0 is None else x0)
        info = capi.pcg(ctx, A, b, x, rtol=rtol, mode=mode, graph=graph, maxit=maxit,
                        raise_on_noconv=False)
        out.append((info, x.numpy()))
        x.close()
    b.close()
    (ia, xa), (ib, xb) = out
    assert ia.converged == ib.converged
    if ia.converged:
        bound = 2.2 * rtol * bn / 1e-3
        assert np.linalg.norm(xa - xb) <= bound, (np.linalg.norm(xa - xb), bound)
    return out


P1 = ((1, 0), (0, 1), (1, 1))


# one workgroup and one line more, tiles of one line and of one column, the
# limits of 1, 3, 5, 7 and 9 cells a thread, the other diagonal, five-point and
# tridiagonal stencils (which have fewer off-diagonals than the kernel holds)
@pytest.mark.parametrize("S, L, steps", [
    (128, 1, ((1, 0),)), (700, 1, ((1, 0),)), (20, 21, P1), (21, 24, P1), (4, 300, P1),
    (1500, 3, P1), (64, 64, ((1, 0), (0, 1))), (65, 65, ((1, 0), (0, 1), (-1, 1))),
    (362, 363, P1), (513, 513, P1), (640, 631, P1), (2049, 257, P1), (1025, 1025, P1),
])
@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("mode", MODES)
def test_resident_pcg_on_a_lattice(ctx, S, L, steps, symmetric, mode):
    r, c, v, n = _lattice_system(S, L, steps, S + L, symmetric)
    A = capi.coo_to_csr(ctx, r, c, v, n, n)
    out = _compare(ctx, A, n, mode, n + 1)
    if capi.solver_storage(A)[0] == capi.STORAGE_DIA:
        assert out[1][0].syncs == 1  # the resident solve ran
    # a nonzero start, and the iteration cap
    x0 = np.random.default_rng(5).standard_normal(n)
    _compare(ctx, A, n, mode, n + 2, x0=x0)
    out = _compare(ctx, A, n, mode, n + 2, x0=x0, maxit=3, rtol=1e-14)
    assert out[0][0].iters == out[1][0].iters == 3
    # three steps of the recurrence: its precision, and the start's rounding
    eps = 1e-13 if mode == capi.PCG_FP64 else 1e-5 if mode == capi.PCG_MIXED else 1e-12
    assert np.linalg.norm(out[0][1] - out[1][1]) <= eps * np.linalg.norm(out[0][1])
    A.close()


# teams of 1, 2, 31 to 33 (one wavefront or two sum the members), 63 to 65 (one
# hop or two) and 256 workgroups: 64 lines of 6 cells each; tolerance as above
@pytest.mark.parametrize("team", [1, 2, 31, 32, 33, 63, 64, 65, 256])
@pytest.mark.parametrize("mode", MODES)
def test_team_sums(ctx, team, mode):
    r, c, v, n = _lattice_system(6, 64 * team, P1, team)
    A = capi.coo_to_csr(ctx, r, c, v, n, n)
    x0 = np.random.default_rng(5).standard_normal(n)
    out = _compare(ctx, A, n, mode, team + 2, x0=x0, maxit=3, rtol=1e-14)
    assert out[0][0].iters == out[1][0].iters == 3
    assert abs(out[0][0].relres - out[1][0].relres) <= 1e-4 * out[0][0].relres
    eps = 1e-13 if mode == capi.PCG_FP64 else 1e-5 if mode == capi.PCG_MIXED else 1e-12
    assert np.linalg.norm(out[0][1] - out[1][1]) <= eps * np.linalg.norm(out[0][1])
    A.close()


# the streamed matrix: 17, 25 and 33 cells a thread
@pytest.mark.parametrize("S, L", [(1141, 1140), (1449, 1448), (1400, 1900), (2049, 2049),
                                  (3000, 500)])
@pytest.mark.parametrize("mode", MODES)
def test_resident_pcg_on_large_lattices(ctx, S, L, mode):
    r, c, v, n = _lattice_system(S, L, P1, 3)
    v[-n:] += 1.0  # well conditioned: a few dozen iterations
    A = capi.coo_to_csr(ctx, r, c, v, n, n)
    out = _compare(ctx, A, n, mode, 4)
    assert out[1][0].syncs == 1 and out[1][0].converged
    A.close()


def test_streamed_lattice_without_a_diagonal_entry_keeps_the_sweeps(ctx):
    # (the streamed solve takes the diagonal from the row sums)
    S, L = 1141, 1140
    r, c, v, n = _lattice_system(S, L, P1, 3)
    k = np.nonzero((r == c) & (r == n // 2))[0]
    r, c, v = (np.delete(q, k) for q in (r, c, v))
    A = capi.coo_to_csr(ctx, r, c, v, n, n)
    out = _compare(ctx, A, n, capi.PCG_FP64, 1, maxit=3, rtol=1e-14)
    assert np.array_equal(out[0][1], out[1][1])  # graph replay against plain launches
    A.close()


@pytest.mark.parametrize("mode", MODES)
def test_resident_pcg_is_deterministic_and_zero_rhs(ctx, mode):
    r, c, v, n = _lattice_system(264, 265, P1, 9)
    A = capi.coo_to_csr(ctx, r, c, v, n, n)
    b, x = capi.Vec(ctx, np.random.default_rng(2).standard_normal(n)), capi.Vec(ctx, n)
    got = []
    for _ in range(3):
        x.fill(0.0)
        capi.pcg(ctx, A, b, x, mode=mode)
        got.append(x.numpy())
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    b.fill(0.0)
    x.fill(2.0)
    info = capi.pcg(ctx, A, b, x, mode=mode)
    assert info.converged and info.iters == 0 and not x.numpy().any()
    for h in (x, b, A):
        h.close()


# sliced ELL: lattices whose squares are cut along random diagonals; fewer rows
# than a slice, one workgroup, teams summed in one and in two hops, 2, 3, 5, 8
# and 11 rows a thread
@pytest.mark.parametrize("S, L", [(7, 8), (22, 23), (40, 64), (181, 182), (363, 362), (450, 451),
                                  (512, 513), (800, 801), (1025, 1024), (1150, 1151)])
@pytest.mark.parametrize("mode", MODES)
def test_resident_pcg_on_ell(ctx, S, L, mode):
    r2, c2, v2, n = _flipped_system(S, L, S)
    A = capi.coo_to_csr(ctx, r2, c2, v2, n, n)
    out = _compare(ctx, A, n, mode, n + 1)
    assert capi.solver_storage(A)[0] == capi.STORAGE_ELL16
    assert out[1][0].syncs == 1  # the resident solve ran
    x0 = np.random.default_rng(5).standard_normal(n)
    out = _compare(ctx, A, n, mode, n + 2, x0=x0, maxit=3, rtol=1e-14)
    assert out[0][0].iters == out[1][0].iters == 3
    eps = 1e-13 if mode == capi.PCG_FP64 else 1e-5 if mode == capi.PCG_MIXED else 1e-12
    assert np.linalg.norm(out[0][1] - out[1][1]) <= eps * np.linalg.norm(out[0][1])
    A.close()


def _kinds_system(S, L, seed):
    """A system with three kinds of rows, numbered kind by kind as third-order
    DOFs are: the lattice's vertices (up to 24 neighbours), two nodes on every
    edge and one in every triangle (three each); weights as _lattice_system."""
    rng = np.random.default_rng(seed)
    v = np.arange(S * L).reshape(L, S)
    e = np.concatenate([np.stack([a.ravel(), b.ravel()], 1) for a, b in (
        (v[:, :-1], v[:, 1:]), (v[:-1], v[1:]), (v[:-1, :-1], v[1:, 1:]))])
    t = np.concatenate([np.stack([c.ravel() for c in k], 1) for k in (
        (v[:-1, :-1], v[:-1, 1:], v[1:, 1:]), (v[:-1, :-1], v[1:, :-1], v[1:, 1:]))])
    one = v.size + 2 * np.arange(len(e))  # an edge's first node
    mid = v.size + 2 * len(e) + np.arange(len(t))
    pairs = np.concatenate([e, np.stack([one, one + 1], 1)]
                           + [np.stack([e[:, k], one + m], 1) for k in (0, 1) for m in (0, 1)]
                           + [np.stack([t[:, k], mid], 1) for k in (0, 1, 2)])
    n = v.size + 2 * len(e) + len(t)
    i, j = pairs.T
    w = np.exp(rng.standard_normal(i.size))
    diag = np.full(n, 1e-3)
    np.add.at(diag, i, w)
    np.add.at(diag, j, w)
    k = np.arange(n)
    return np.concatenate([i, j, k]), np.concatenate([j, i, k]), np.concatenate([-w, -w, diag]), n


# rows of several lengths: one part, parts with their share of every length
# (one to three rows a thread, rows longer than what stays in registers) and
# runs of rows
@pytest.mark.parametrize("S, L", [(5, 4), (12, 10), (40, 41), (130, 129), (160, 150), (200, 190),
                                  (230, 220)])
@pytest.mark.parametrize("mode", MODES)
def test_resident_pcg_on_rows_of_several_lengths(ctx, S, L, mode):
    r, c, v, n = _kinds_system(S, L, S)
    A = capi.coo_to_csr(ctx, r, c, v, n, n)
    out = _compare(ctx, A, n, mode, n + 1)
    assert capi.solver_storage(A)[0] == capi.STORAGE_ELL16 and out[1][0].syncs == 1
    x0 = np.random.default_rng(5).standard_normal(n)
    out = _compare(ctx, A, n, mode, n + 2, x0=x0, maxit=3, rtol=1e-14)
    assert out[0][0].iters == out[1][0].iters == 3
    eps = 1e-13 if mode == capi.PCG_FP64 else 1e-5 if mode == capi.PCG_MIXED else 1e-12
    assert np.linalg.norm(out[0][1] - out[1][1]) <= eps * np.linalg.norm(out[0][1])
    A.close()


def test_wrapped_band_matrix_keeps_the_sweeps(ctx):
    # the offsets of a lattice, but entries across the lines' ends
    n, S = 4096, 64
    i = np.arange(n)
    rows, cols, vals = [i], [i], [np.full(n, 7.0)]
    for o in (1, S, S + 1):
        rows += [i[:-o], i[o:]]
        cols += [i[o:], i[:-o]]
        vals += [np.full(n - o, -1.0)] * 2
    A = capi.coo_to_csr(ctx, np.concatenate(rows), np.concatenate(cols), np.concatenate(vals), n, n)
    out = _compare(ctx, A, n, capi.PCG_FP64, 1)
    assert np.array_equal(out[0][1], out[1][1])  # graph replay against plain launches
    A.close()


# more teams than the chip holds at once, 5 x 5 to 90 x 90 problems and in FP64
# single rows (on which the reliable updates fail: the one step exhausts the
# Krylov space, and the old direction that they keep is no longer conjugate);
# all lattices, none, and both (which take a launch each)
@pytest.mark.parametrize("kind", ["lattice", "flipped", "both"])
@pytest.mark.parametrize("mode", MODES)
def test_resident_batch(ctx, kind, mode):
    rng = np.random.default_rng(17)
    parts, off = [], [0]
    for k in range(300):
        S, L = (int(q) for q in rng.integers(5, 60 if k else 91, 2))
        if k % 50 == 7 and mode == capi.PCG_FP64:
            r, c, v, n = np.array([0]), np.array([0]), np.array([2.0]), 1
        elif kind == "lattice" or (kind == "both" and k % 3):
            r, c, v, n = _lattice_system(S, L, P1, k)
        else:
            r, c, v, n = _flipped_system(S, L, k)
        parts.append((r + off[-1], c + off[-1], v))
        off.append(off[-1] + n)
    n = off[-1]
    A = capi.coo_to_csr(ctx, *(np.concatenate(p) for p in zip(*parts)), n, n)
    bh = rng.standard_normal(n)
    bh[off[3]:off[4]] = 0.0  # a zero right-hand side
    b = capi.Vec(ctx, bh)
    batch = capi.Batch(ctx, A, np.array(off, np.int32))
    out = []
    for graph in (1, 0, 0):
        x = capi.Vec(ctx, np.ones(n))
        summ, infos = batch.pcg(b, x, rtol=1e-10, maxit=20000, mode=mode, graph=graph)
        out.append((summ, infos, x.numpy()))
        x.close()
    assert all(s.converged for s, _, _ in out)
    assert out[1][0].syncs == 1  # the resident solve ran
    assert np.array_equal(out[1][2], out[2][2])
    assert out[1][1][3].iters == 0 and not out[1][2][off[3]:off[4]].any()
    for k in range(300):
        xa, xb = (o[2][off[k]:off[k + 1]] for o in out[:2])
        bound = 2.2e-10 * np.linalg.norm(bh[off[k]:off[k + 1]]) / 1e-3
        assert np.linalg.norm(xa - xb) <= bound, k
    for h in (batch, b, A):
        h.close()


# a problem of more rows than two a thread hold beside a small one (the kernel
# of eight rows a thread), and problems that the small kernel takes in turns
@pytest.mark.parametrize("make", [
    lambda: [_flipped_system(520, 521, 1), _kinds_system(40, 41, 2)],
    lambda: [_kinds_system(70 + k, 60, k) for k in range(12)],
])
@pytest.mark.parametrize("mode", MODES)
def test_resident_batch_of_large_problems(ctx, make, mode):
    parts, off = [], [0]
    for r, c, v, n in make():
        parts.append((r + off[-1], c + off[-1], v))
        off.append(off[-1] + n)
    n = off[-1]
    A = capi.coo_to_csr(ctx, *(np.concatenate(p) for p in zip(*parts)), n, n)
    bh = np.random.default_rng(3).standard_normal(n)
    b = capi.Vec(ctx, bh)
    batch = capi.Batch(ctx, A, np.array(off, np.int32))
    out = []
    for graph in (1, 0):
        x = capi.Vec(ctx, n)
        summ, _ = batch.pcg(b, x, rtol=1e-10, maxit=20000, mode=mode, graph=graph)
        assert summ.converged
        out.append(x.numpy())
        x.close()
    assert summ.syncs == 1  # the resident solve ran
    for lo, hi in zip(off, off[1:]):
        bound = 2.2e-10 * np.linalg.norm(bh[lo:hi]) / 1e-3
        assert np.linalg.norm(out[0][lo:hi] - out[1][lo:hi]) <= bound
    for h in (batch, b, A):
        h.close()


def _fixed_band(system, first, last):
    """The system with rows first..last - 1 fixed (identity rows and columns)."""
    r, c, v, n = system
    fixed = np.zeros(n, bool)
    fixed[first:last] = True
    keep = (~fixed[r] & ~fixed[c]) | (r == c)
    r, c, v = r[keep], c[keep], v[keep].copy()
    v[(r == c) & fixed[r]] = 1.0
    return r, c, v, n


def _turned_lattice(S, L, at, seed):
    """_lattice_system whose squares below line `at` are cut along the other
    diagonal."""
    y = np.arange(L * S) // S
    r, c, v, n = _lattice_system(S, L, ((1, 0), (0, 1), (1, 1)), seed)
    r2, c2, v2, _ = _lattice_system(S, L, ((1, 0), (0, 1), (-1, 1)), seed + 1)
    keep = (abs(r - c) != S + 1) | (np.minimum(y[r], y[c]) >= at)
    turn = (abs(r2 - c2) == S - 1) & (np.minimum(y[r2], y[c2]) < at)
    r, c, v = (np.concatenate([a[keep], b[turn]]) for a, b in ((r, r2), (c, c2), (v, v2)))
    off = r != c
    v[~off] = 1e-3
    diag = np.zeros(n)
    np.subtract.at(diag, r[off], v[off])
    v[~off] += diag[r[~off]]
    return r, c, v, n


# problems with couplings that the 64 rows from the middle on do not show:
# another diagonal in a part of the lattice, and fixed rows all over the middle
# (a line, and lines of a lattice); beside them a problem with all six
@pytest.mark.parametrize("make", [
    lambda: [_turned_lattice(81, 81, 20, 1), _lattice_system(20, 30, P1, 2)],
    lambda: [_turned_lattice(81, 81, 70, 3), _turned_lattice(100, 12, 3, 4)],
    lambda: [_fixed_band(_lattice_system(400, 1, ((1, 0),), 5), 190, 275),
             _flipped_system(30, 31, 6)],
    lambda: [_fixed_band(_lattice_system(90, 40, P1, 7), 1790, 1890), _flipped_system(30, 31, 8),
             _fixed_band(_lattice_system(300, 1, ((1, 0),), 9), 140, 220),
             _lattice_system(20, 30, P1, 2)],
])
@pytest.mark.parametrize("mode", MODES)
def test_resident_batch_with_couplings_away_from_the_middle(ctx, make, mode):
    parts, off = [], [0]
    for r, c, v, n in make():
        parts.append((r + off[-1], c + off[-1], v))
        off.append(off[-1] + n)
    n = off[-1]
    A = capi.coo_to_csr(ctx, *(np.concatenate(p) for p in zip(*parts)), n, n)
    bh = np.random.default_rng(3).standard_normal(n)
    b = capi.Vec(ctx, bh)
    batch = capi.Batch(ctx, A, np.array(off, np.int32))
    out = []
    for graph in (-1, 0):
        x = capi.Vec(ctx, n)
        summ, _ = batch.pcg(b, x, rtol=1e-10, maxit=20000, mode=mode, graph=graph)
        assert summ.converged
        out.append(x.numpy())
        x.close()
    assert summ.syncs == 1  # the resident solve ran
    for lo, hi in zip(off, off[1:]):
        bound = 2.2e-10 * np.linalg.norm(bh[lo:hi]) / 1e-3
        assert np.linalg.norm(out[0][lo:hi] - out[1][lo:hi]) <= bound
    for h in (batch, b, A):
        h.close()


# a context whose resident solves give up their waits at once: the flag is up
# from the start, whatever the workgroup that reports the outcome has seen, and
# the sweeps go on; one workgroup, one hop, two hops, the streamed matrix, the
# three kernels on sliced ELL; then a solve on the same words and a fresh one
@pytest.mark.parametrize("make", [
    lambda: _lattice_system(20, 21, P1, 1), lambda: _lattice_system(65, 65, P1, 2),
    lambda: _lattice_system(362, 363, P1, 3), lambda: _lattice_system(1141, 1140, P1, 3),
    lambda: _flipped_system(40, 64, 4), lambda: _flipped_system(450, 451, 5),
    lambda: _kinds_system(130, 129, 6),
])
@pytest.mark.parametrize("mode", MODES)
def test_solve_that_gives_up_its_waits_ends_in_the_sweeps(make, mode):
    r, c, v, n = make()
    if n > 10**6:
        v[-n:] += 1.0
    bh = np.random.default_rng(1).standard_normal(n)
    bound = 2.2e-10 * np.linalg.norm(bh) / 1e-3
    with capi.Context(0) as ctx:
        A, fresh = (capi.coo_to_csr(ctx, r, c, v, n, n) for _ in range(2))
        b, x = capi.Vec(ctx, bh), capi.Vec(ctx, n)
        capi.pcg(ctx, A, b, x, mode=mode, graph=-1)
        want = x.numpy()
        x.fill(0.0)
        ctx.set_resident_wait(0.0)
        info = capi.pcg(ctx, A, b, x, rtol=1e-10, mode=mode)
        assert info.converged and info.syncs >= 2
        assert np.linalg.norm(x.numpy() - want) <= bound
        ctx.set_resident_wait(4.0)
        for M in (A, fresh):
            x.fill(0.0)
            info = capi.pcg(ctx, M, b, x, rtol=1e-10, mode=mode)
            assert info.converged and (info.syncs == 1 or M is A)
            assert np.linalg.norm(x.numpy() - want) <= bound
        for h in (x, b, A, fresh):
            h.close()


@pytest.mark.parametrize("kind", ["lattice", "flipped", "both"])
@pytest.mark.parametrize("mode", MODES)
def test_batch_that_gives_up_its_waits_ends_in_the_sweeps(kind, mode):
    parts, off = [], [0]
    for k in range(12):
        make = _flipped_system if kind == "flipped" or (kind == "both" and k % 2) else (
            lambda S, L, seed: _lattice_system(S, L, P1, seed))
        r, c, v, n = make(20 + 11 * k, 30 + 5 * k, k)
        parts.append((r + off[-1], c + off[-1], v))
        off.append(off[-1] + n)
    n = off[-1]
    bh = np.random.default_rng(3).standard_normal(n)
    with capi.Context(0) as ctx:
        A = capi.coo_to_csr(ctx, *(np.concatenate(p) for p in zip(*parts)), n, n)
        b, x = capi.Vec(ctx, bh), capi.Vec(ctx, n)
        out = []
        for graph, seconds in ((-1, 4.0), (0, 0.0), (0, 4.0)):
            batch = capi.Batch(ctx, A, np.array(off, np.int32))
            ctx.set_resident_wait(seconds)
            x.fill(0.0)
            summ, infos = batch.pcg(b, x, rtol=1e-10, maxit=20000, mode=mode, graph=graph)
            assert summ.converged and all(i.converged for i in infos)
            out.append((summ.syncs, x.numpy()))
            batch.close()
        assert out[1][0] >= 2 and out[2][0] == 1
        for lo, hi in zip(off, off[1:]):
            bound = 2.2e-10 * np.linalg.norm(bh[lo:hi]) / 1e-3
            for _, got in out[1:]:
                assert np.linalg.norm(got[lo:hi] - out[0][1][lo:hi]) <= bound
        for h in (x, b, A):
            h.close()


def test_resident_wait_is_checked(ctx):
    for bad in (-1.0, float("nan")):
        with pytest.raises(capi.LfgpuError) as e:
            ctx.set_resident_wait(bad)
        assert e.value.code == capi.EINVAL


# problems that take more than half of the chip each, one after the other: the
# workgroups that are first at the second one wait for the rest of its team
# until the first problem is done, several times the bound of a wait here
@pytest.mark.parametrize("make", [lambda k: _lattice_system(840, 830, P1, k),
                                  lambda k: _flipped_system(800, 801, k)])
def test_batch_waits_for_a_team_as_long_as_the_problem_before_takes(make):
    parts, off, maxit = [], [0], 8000
    for k in range(2):
        r, c, v, n = make(k)
        parts.append((r + off[-1], c + off[-1], v))
        off.append(off[-1] + n)
    n = off[-1]
    with capi.Context(0) as ctx:
        A = capi.coo_to_csr(ctx, *(np.concatenate(p) for p in zip(*parts)), n, n)
        b, x = capi.Vec(ctx, np.random.default_rng(3).standard_normal(n)), capi.Vec(ctx, n)
        batch = capi.Batch(ctx, A, np.array(off, np.int32))
        batch.pcg(b, x, rtol=0.0, maxit=2, raise_on_noconv=False)  # (builds the plans)
        ctx.set_resident_wait(0.012)
        summ, infos = batch.pcg(b, x, rtol=0.0, maxit=maxit, raise_on_noconv=False)
        assert summ.syncs == 1 and all(i.iters == maxit for i in infos)
        assert summ.ms > 2 * 2 * 12.0  # (else the bound was not reached)
        for h in (batch, x, b, A):
            h.close()


def test_small_unstructured_problems_take_little_memory():
    # 3000 problems of 64 rows, which read no rows of other workgroups
    total, now = ctypes.c_size_t(), ctypes.c_size_t()

    def free_bytes():
        assert capi.lib().hipMemGetInfo(ctypes.byref(now), ctypes.byref(total)) == 0
        return now.value

    parts, off = [], [0]
    for k in range(3000):
        r, c, v, n = _flipped_system(8, 8, k)
        parts.append((r + off[-1], c + off[-1], v))
        off.append(off[-1] + n)
    n = off[-1]
    with capi.Context(0) as ctx:
        A = capi.coo_to_csr(ctx, *(np.concatenate(p) for p in zip(*parts)), n, n)
        b, x = capi.Vec(ctx, np.random.default_rng(3).standard_normal(n)), capi.Vec(ctx, n)
        batch = capi.Batch(ctx, A, np.array(off, np.int32))
        free = []
        for graph in (1, 0):
            x.fill(0.0)
            summ, _ = batch.pcg(b, x, graph=graph)
            free.append(free_bytes())
        assert summ.syncs == 1  # the resident solve ran
        # its matrix (10 B a slot), places (2 B a slot), team sums (10 KB a
        # problem of one workgroup at most) and vectors
        assert free[0] - free[1] < 64 << 20, free
        for h in (batch, x, b, A):
            h.close()


@pytest.mark.parametrize("mode", MODES)
def test_resident_solves_come_back_after_one_that_gave_up(mode):
    r, c, v, n = _flipped_system(60, 61, 1)
    with capi.Context(0) as ctx:
        A = capi.coo_to_csr(ctx, r, c, v, n, n)
        batch = capi.Batch(ctx, A, np.array([0, n], np.int32))
        b, x = capi.Vec(ctx, np.random.default_rng(1).standard_normal(n)), capi.Vec(ctx, n)

        def batched(*a, **k):
            return batch.pcg(*a, **k)[0]
        for solve in (batched, lambda *a, **k: capi.pcg(ctx, A, *a, **k)):
            for seconds in (0.0, 4.0, 0.0, 0.0, 4.0):
                # (the sweeps take the next calls for 16, then 32 times what the
                # lost launches took, a few ms each)
                time.sleep(0.3)
                ctx.set_resident_wait(seconds)
                x.fill(0.0)
                info = solve(b, x, rtol=1e-10, mode=mode)
                assert info.converged and (info.syncs == 1) == (seconds > 0.0)
        for h in (x, b, batch, A):
            h.close()


# a call on a new batch finds the rows' order and splits them over teams: that
# takes less than the sweeps' own first call (which tunes and captures) and their
# solve
@pytest.mark.parametrize("S, count", [(8, 20000), (64, 1000)])
def test_first_call_on_unstructured_problems(ctx, S, count):
    some = [_flipped_system(S, S, k) for k in range(8)]
    n = some[0][3]
    parts = [(r + k * n, c + k * n, v) for k in range(count) for r, c, v, _ in (some[k % 8],)]
    A = capi.coo_to_csr(ctx, *(np.concatenate(p) for p in zip(*parts)), n * count, n * count)
    bh = np.random.default_rng(3).standard_normal((count, n))
    b, x = capi.Vec(ctx, bh), capi.Vec(ctx, n * count)
    off = np.arange(count + 1, dtype=np.int32) * n
    best, got = {}, {}
    for graph in (1, 0, 1, 0, 1, 0):
        batch = capi.Batch(ctx, A, off)
        x.fill(0.0)
        ctx.sync()
        start = time.perf_counter()
        batch.pcg(b, x, rtol=1e-10, graph=graph)
        best[graph] = min(best.get(graph, 1e9), time.perf_counter() - start)
        got[graph] = x.numpy().reshape(count, n)
        batch.close()
    assert best[0] <= 1.3 * best[1], best  # (0.4 to 0.7; 1.8 and 2.8 with a sort on the host)
    bound = 2.2e-10 * np.linalg.norm(bh, axis=1) / 1e-3
    assert (np.linalg.norm(got[0] - got[1], axis=1) <= bound).all()
    for h in (x, b, A):
        h.close()


# a line and a row that couples to all: the first call, which gives every slot its
# place, takes no longer than the sweeps' first call, also where that row does not
# fit a workgroup
@pytest.mark.parametrize("n, fits", [(20000, True), (32000, False)])
def test_first_call_on_a_matrix_with_a_long_row(ctx, n, fits):
    i = np.arange(1, n)
    w = np.exp(np.random.default_rng(1).standard_normal(2 * n - 3))
    r, c = np.concatenate([np.zeros(n - 1, np.int64), i[:-1]]), np.concatenate([i, i[1:]])
    diag = np.full(n, 1e-1)
    np.add.at(diag, r, w)
    np.add.at(diag, c, w)
    k = np.arange(n)
    bh = np.random.default_rng(2).standard_normal(n)
    b, x = capi.Vec(ctx, bh), capi.Vec(ctx, n)
    best, got = {}, {}
    for graph in (1, 0, 1, 0, 1, 0):
        A = capi.coo_to_csr(ctx, np.concatenate([r, c, k]), np.concatenate([c, r, k]),
                            np.concatenate([-w, -w, diag]), n, n)
        x.fill(0.0)
        ctx.sync()
        start = time.perf_counter()
        info = capi.pcg(ctx, A, b, x, rtol=1e-10, graph=graph)
        best[graph] = min(best.get(graph, 1e9), time.perf_counter() - start)
        assert info.converged and (graph == 1 or (info.syncs == 1) == fits)
        got[graph] = x.numpy()
        A.close()
    assert best[0] <= 1.15 * best[1], best  # (0.6 and 1.0; 1.4 and 1.2 with searches)
    assert np.linalg.norm(got[0] - got[1]) <= 2.2e-10 * np.linalg.norm(bh) / 0.1
    for h in (x, b):
        h.close()


# many small lattices: the first call plans for its own mode only, and another
# mode's first call for that one
def test_first_call_on_many_lattices(ctx):
    S, count = 9, 40000
    some = [_lattice_system(S, S, P1, k) for k in range(8)]
    n = some[0][3]
    parts = [(r + k * n, c + k * n, v) for k in range(count) for r, c, v, _ in (some[k % 8],)]
    A = capi.coo_to_csr(ctx, *(np.concatenate(p) for p in zip(*parts)), n * count, n * count)
    bh = np.random.default_rng(3).standard_normal((count, n))
    b, x = capi.Vec(ctx, bh), capi.Vec(ctx, n * count)
    off = np.arange(count + 1, dtype=np.int32) * n
    got, free, total, now = [], [], ctypes.c_size_t(), ctypes.c_size_t()
    batch = capi.Batch(ctx, A, off)
    for graph in (1, 0):
        x.fill(0.0)
        summ, _ = batch.pcg(b, x, rtol=1e-10, graph=graph)
        assert capi.lib().hipMemGetInfo(ctypes.byref(now), ctypes.byref(total)) == 0
        free.append(now.value)
    assert summ.syncs == 1  # the resident solve ran
    # one plan: 120 B of a job, 8 of a slot and 4 of a counter a problem, and the
    # outcomes' 32 B (three plans take 12 MB more)
    assert free[0] - free[1] < 12 << 20, free
    got.append(x.numpy().reshape(count, n))
    for mode in (capi.PCG_MIXED_MATRIX, capi.PCG_FP64):
        x.fill(0.0)
        batch.pcg(b, x, rtol=1e-10, mode=mode)
        got.append(x.numpy().reshape(count, n))
    assert np.array_equal(got[0], got[2])
    bound = 2.2e-10 * np.linalg.norm(bh, axis=1) / 1e-3
    assert (np.linalg.norm(got[0] - got[1], axis=1) <= bound).all()
    for h in (batch, x, b, A):
        h.close()


# many small lattices in the mixed modes, where the sweeps are faster and run;
# FP64 stays in one launch
@pytest.mark.parametrize("mode", MODES)
def test_many_small_lattices(ctx, mode):
    S, count = 8, 20000
    some = [_lattice_system(S, S, P1, k) for k in range(8)]
    n = some[0][3]
    parts = [(r + k * n, c + k * n, v) for k in range(count) for r, c, v, _ in (some[k % 8],)]
    A = capi.coo_to_csr(ctx, *(np.concatenate(p) for p in zip(*parts)), n * count, n * count)
    bh = np.random.default_rng(3).standard_normal((count, n))
    b, x = capi.Vec(ctx, bh), capi.Vec(ctx, n * count)
    batch = capi.Batch(ctx, A, np.arange(count + 1, dtype=np.int32) * n)
    got = {}
    for graph in (1, 0, 0):
        x.fill(0.0)
        summ, _ = batch.pcg(b, x, rtol=1e-10, mode=mode, graph=graph)
        assert graph == 1 or (summ.syncs == 1) == (mode == capi.PCG_FP64)
        got[graph] = x.numpy().reshape(count, n)
    bound = 2.2e-10 * np.linalg.norm(bh, axis=1) / 1e-3
    assert (np.linalg.norm(got[0] - got[1], axis=1) <= bound).all()
    for h in (batch, x, b, A):
        h.close()


def test_lattices_of_one_workgroup_take_no_words():
    # 20000 problems of 25 rows, which exchange nothing with other workgroups
    parts, off = [], [0]
    for k in range(20000):
        r, c, v, n = _lattice_system(5, 5, P1, k) if k < 4 else parts[k % 4]
        parts.append((r, c, v, n))
        off.append(off[-1] + n)
    n = off[-1]
    trip = [(r + o, c + o, v) for (r, c, v, _), o in zip(parts, off)]
    total, now = ctypes.c_size_t(), ctypes.c_size_t()
    with capi.Context(0) as ctx:
        A = capi.coo_to_csr(ctx, *(np.concatenate(p) for p in zip(*trip)), n, n)
        b, x = capi.Vec(ctx, np.random.default_rng(3).standard_normal(n)), capi.Vec(ctx, n)
        batch = capi.Batch(ctx, A, np.array(off, np.int32))
        free = []
        for graph in (1, 0):
            x.fill(0.0)
            summ, _ = batch.pcg(b, x, graph=graph)
            assert capi.lib().hipMemGetInfo(ctypes.byref(now), ctypes.byref(total)) == 0
            free.append(now.value)
        assert summ.syncs == 1  # the resident solve ran
        # jobs, slots and outcomes: 200 B a problem
        assert free[0] - free[1] < 16 << 20, free
        for h in (batch, x, b, A):
            h.close()


# a few large unstructured problems, more than the chip holds at once: in the
# FP32-Krylov mode the sweeps are faster
def test_few_large_unstructured_problems(ctx):
    parts, off = [], [0]
    for k in range(2):
        r, c, v, n = _flipped_system(760, 761, k)
        parts.append((r + off[-1], c + off[-1], v))
        off.append(off[-1] + n)
    n = off[-1]
    A = capi.coo_to_csr(ctx, *(np.concatenate(p) for p in zip(*parts)), n, n)
    b, x = capi.Vec(ctx, np.random.default_rng(3).standard_normal(n)), capi.Vec(ctx, n)
    batch = capi.Batch(ctx, A, np.array(off, np.int32))
    for mode in MODES:
        summ, _ = batch.pcg(b, x, maxit=300, mode=mode, raise_on_noconv=False)
        assert (summ.syncs == 1) == (mode != capi.PCG_MIXED)
    for h in (batch, x, b, A):
        h.close()


# entries (of value zero) on one side only: a workgroup then reads rows of others
# that read none of its own; one to three rows a thread, five, and eight
@pytest.mark.parametrize("S, L", [(40, 64), (181, 182), (363, 362), (512, 513), (800, 801),
                                  (1025, 1024)])
@pytest.mark.parametrize("mode", MODES)
def test_resident_pcg_on_an_unsymmetric_pattern(ctx, S, L, mode):
    r, c, v, n = _flipped_system(S, L, S)
    rng = np.random.default_rng(S)
    i = rng.integers(0, n // 2, n // 4)  # the upper half reads ahead
    j = np.minimum(i + rng.integers(2, 3 * S, i.size), n - 1)
    A = capi.coo_to_csr(ctx, np.concatenate([r, i]), np.concatenate([c, j]),
                        np.concatenate([v, np.zeros(i.size)]), n, n)
    out = _compare(ctx, A, n, mode, n + 1)
    assert capi.solver_storage(A)[0] == capi.STORAGE_ELL16 and out[1][0].syncs == 1
    x0 = np.random.default_rng(5).standard_normal(n)
    out = _compare(ctx, A, n, mode, n + 2, x0=x0, maxit=3, rtol=1e-14)
    assert out[0][0].iters == out[1][0].iters == 3
    eps = 1e-13 if mode == capi.PCG_FP64 else 1e-5 if mode == capi.PCG_MIXED else 1e-12
    assert np.linalg.norm(out[0][1] - out[1][1]) <= eps * np.linalg.norm(out[0][1])
    A.close()


# the three modes in turn on one matrix (other teams and layouts in the same
# words), with caps that use up the exchanges' numbers, so that the words are
# cleared, and with small ones: every solve like the first of its mode on a matrix
# of its own
@pytest.mark.parametrize("make", [
    lambda: _lattice_system(65, 65, P1, 2), lambda: _lattice_system(362, 363, P1, 3),
    lambda: _flipped_system(40, 64, 4), lambda: _flipped_system(363, 362, 5),
])
def test_resident_solves_share_their_words(ctx, make):
    r, c, v, n = make()
    A = capi.coo_to_csr(ctx, r, c, v, n, n)
    batch = capi.Batch(ctx, A, np.array([0, n], np.int32))
    b, x = capi.Vec(ctx, np.random.default_rng(1).standard_normal(n)), capi.Vec(ctx, n)
    for call in (lambda M, B, **k: capi.pcg(ctx, M, b, x, **k),
                 lambda M, B, **k: B.pcg(b, x, **k)[0]):
        want = {}
        for maxit in (20000, 2**31 - 1, 20000, 6 * 10**8, 6 * 10**8, 2**31 - 1):
            for mode in MODES:
                if mode not in want:
                    M = capi.coo_to_csr(ctx, r, c, v, n, n)
                    B = capi.Batch(ctx, M, np.array([0, n], np.int32))
                    x.fill(0.0)
                    call(M, B, mode=mode, maxit=20000)
                    want[mode] = x.numpy()
                    B.close()
                    M.close()
                x.fill(0.0)
                info = call(A, batch, mode=mode, maxit=maxit)
                assert info.converged and info.syncs == 1
                assert np.array_equal(x.numpy(), want[mode])
    for h in (batch, x, b, A):
        h.close()


# the streamed FP64 solve updates x in memory, the last time perhaps by a sum
# that a workgroup took for whole: where it gives up, the sweeps begin at the
# caller's x
def test_streamed_solve_that_gives_up_leaves_the_start(ctx):
    r, c, v, n = _lattice_system(1141, 1140, P1, 3)
    v[-n:] += 1.0
    start = np.random.default_rng(2).standard_normal(n)
    with capi.Context(0) as own:
        A = capi.coo_to_csr(own, r, c, v, n, n)
        b = capi.Vec(own, np.random.default_rng(1).standard_normal(n))
        x = capi.Vec(own, start)
        swept = capi.pcg(own, A, b, x, graph=-1)
        want = x.numpy()
        own.set_resident_wait(0.0)
        x.upload(start)
        info = capi.pcg(own, A, b, x)
        assert info.syncs >= 2 and info.iters == swept.iters
        assert np.array_equal(x.numpy(), want)
        for h in (x, b, A):
            h.close()
