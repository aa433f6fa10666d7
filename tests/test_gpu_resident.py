"""The resident solves (lfgpu_resident.hip) against the two-sweep solver.

opts->graph = -1 runs the sweeps, 0 (the default) the resident solve where
the system fits the chip.  Both run the same recurrences and stop on the same
test with sums in another order.  Iteration counts: a solve of k iterations
to rtol 1e-10 gains ln(1e10) / k an iteration on average, and the residual
norm oscillates about that trend by tens of percent, at places that rounding
moves: 2 % of k (at least 2) is a factor of 1.6 in the residual.  Solutions to
100 rtol: each is within about kappa(D^-1 A)^(1/2) rtol of the exact one in
the energy norm, and the measured errors of such solves against direct ones
stay below 20 rtol.
"""
import numpy as np
import pytest

from lehrfempp_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with capi.Context(0) as c:
        yield c


def _band_system(n, offs, seed, symmetric=True):
    """Triplets of a diagonally dominant matrix with the given off-diagonal
    offsets, values random, a reaction term that makes it positive definite."""
    rng = np.random.default_rng(seed)
    rows, cols, vals, diag = [], [], [], np.full(n, 1e-3)
    for o in offs:
        if o >= n:
            continue
        i = np.arange(n - o)
        w = np.exp(rng.standard_normal(n - o))
        rows += [i, i + o]
        cols += [i + o, i]
        vals += [-w, -w if symmetric else -w * (1.0 + 1e-15 * rng.integers(0, 2, n - o))]
        diag[: n - o] += w
        diag[o:] += w
    rows.append(np.arange(n))
    cols.append(np.arange(n))
    vals.append(diag)
    return np.concatenate(rows), np.concatenate(cols), np.concatenate(vals)


def _compare(ctx, A, n, mode, seed, x0=None, maxit=None, rtol=1e-10):
    b = capi.Vec(ctx, np.random.default_rng(seed).standard_normal(n))
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
    assert abs(ia.iters - ib.iters) <= max(2, 0.02 * ia.iters), (ia.iters, ib.iters)
    assert np.linalg.norm(xa - xb) <= 100 * rtol * np.linalg.norm(xa)
    return out


# rows at the edges of the workgroup's and the team's splits: one workgroup
# (n <= 512), one row more, rows per thread 1, 3, 5, 9 and their limits,
# offsets as long as a workgroup's rows
@pytest.mark.parametrize("n, offs", [
    (128, (1,)), (511, (1, 20)), (512, (1, 20, 21)), (513, (1, 20, 21)), (1537, (1, 700)),
    (4096, (1, 511, 512)), (5000, (1, 512, 513)), (131072, (1, 362, 363)),
    (131073, (1, 362, 363)), (393217, (1, 1535, 1536)), (400000, (2, 1999, 2001)),
])
@pytest.mark.parametrize("symmetric", [True, False])
def test_resident_pcg_on_dia(ctx, n, offs, symmetric):
    r, c, v = _band_system(n, offs, n, symmetric)
    A = capi.coo_to_csr(ctx, r, c, v, n, n)
    out = _compare(ctx, A, n, capi.PCG_FP64, n + 1)
    if capi.solver_storage(A)[0] == capi.STORAGE_DIA:  # (one case pads too much for DIA)
        assert out[1][0].syncs == 1  # the resident solve ran
    # a nonzero start, and the iteration cap
    x0 = np.random.default_rng(5).standard_normal(n)
    _compare(ctx, A, n, capi.PCG_FP64, n + 2, x0=x0)
    out = _compare(ctx, A, n, capi.PCG_FP64, n + 2, x0=x0, maxit=3, rtol=1e-14)
    assert out[0][0].iters == out[1][0].iters == 3
    assert np.linalg.norm(out[0][1] - out[1][1]) <= 1e-13 * np.linalg.norm(out[0][1])
    A.close()


# the streamed matrix: rows per thread 17 and 33, the last with the shared halo
@pytest.mark.parametrize("n, offs", [
    (1300000, (1, 1140, 1141)), (2097152, (1, 1448, 1449)), (2300001, (1, 1516, 1517)),
    (4198401, (1, 2049, 2050)),
])
def test_resident_pcg_on_large_dia(ctx, n, offs):
    r, c, v = _band_system(n, offs, 3)
    v = v.copy()
    v[-n:] += 1.0  # well conditioned: a few dozen iterations
    A = capi.coo_to_csr(ctx, r, c, v, n, n)
    out = _compare(ctx, A, n, capi.PCG_FP64, 4)
    assert out[1][0].syncs == 1 and out[1][0].converged
    A.close()


def test_resident_pcg_is_deterministic_and_zero_rhs(ctx):
    n = 70000
    r, c, v = _band_system(n, (1, 264, 265), 9)
    A = capi.coo_to_csr(ctx, r, c, v, n, n)
    b, x = capi.Vec(ctx, np.random.default_rng(2).standard_normal(n)), capi.Vec(ctx, n)
    got = []
    for _ in range(3):
        x.fill(0.0)
        capi.pcg(ctx, A, b, x)
        got.append(x.numpy())
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    b.fill(0.0)
    x.fill(2.0)
    info = capi.pcg(ctx, A, b, x)
    assert info.converged and info.iters == 0 and not x.numpy().any()
    for h in (x, b, A):
        h.close()
