"""Partial solve jobs on right-hand sides with an infinite entry: an entry
that does not depend on it keeps its finite value, in the block of pivots that
holds it too, and the other right-hand sides are as without it. Against a
plain substitution with the exported factor."""
import numpy as np
import pytest

from tests.conftest import gpu_available
from tests.helpers import dense_front_problem

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no GPU", allow_module_level=True)

from opt_solver_amd import generators as g  # noqa: E402
from opt_solver_amd.solver import SOLVE_BACKWARD, SOLVE_FORWARD, Plan, analyse  # noqa: E402
from tests.test_gpu_edges import block_chains  # noqa: E402


def substitute(e, y, unit, backward):
    """L y' = y or L^T y' = y with the exported factor, entry by entry."""
    y = y.copy()
    fronts = [tuple(int(v) for v in s) for s in e["steps"]]
    with np.errstate(invalid="ignore", over="ignore"):
        for ro, fo, p, f in (reversed(fronts) if backward else fronts):
            rows = e["row_indices"][ro:ro + f]
            L = e["factor_values"][fo:fo + f * p].reshape(p, f)  # L[c]: column c
            for c in (range(p - 1, -1, -1) if backward else range(p)):
                if backward:
                    for i in range(f - 1, c, -1):
                        y[rows[c]] -= L[c, i] * y[rows[i]]
                    if not unit:
                        y[rows[c]] /= L[c, c]
                else:
                    if not unit:
                        y[rows[c]] /= L[c, c]
                    y[rows[c + 1:]] -= L[c, c + 1:, None] * y[rows[c]]
    return y


def check(fac, perm, unit, at, seed):
    n = perm.size
    assert fac.status == 0 and fac.info.two_by_two_pivots == 0  # entry by entry: 1x1 pivots
    e = fac.export()
    inv = np.empty(n, np.int64)
    inv[perm] = np.arange(n)
    Y = np.random.default_rng(seed).uniform(-1, 1, (n, 5))
    Y[at, 0] = np.inf
    for backward in (False, True):
        want = substitute(e, Y, unit, backward)
        assert np.isfinite(want[:, 0]).any() and np.isfinite(want[:, 1:]).all()
        for nr in (1, 3, 5):
            if backward:
                got = fac.solve(Y[:, :nr], SOLVE_BACKWARD)[perm]
            else:
                got = fac.solve(Y[inv][:, :nr], SOLVE_FORWARD)
            fin = np.isfinite(want[:, :nr])
            assert np.array_equal(np.isfinite(got), fin), (backward, nr)
            assert np.abs(got[fin] - want[:, :nr][fin]).max() < 1e-12, (backward, nr)


def dominant(n, seed, spd):
    M = np.random.default_rng([n, seed]).uniform(0.1, 1, (n, n))
    M = M + M.T
    return M + np.diag(2.0 * n * np.where(np.arange(n) % 3 == 0, 1.0 if spd else -1.0, 1.0))


@pytest.mark.parametrize("p,q", [(20, 30), (64, 400), (64, 600), (100, 40), (200, 60), (257, 30)])
def test_indefinite_dense(p, q):
    """Pivots in the middle of a 16-, 64- and 256-column block, the rows below
    in the same workgroup and in others. L's entries are at most about 1 / n,
    so both substitutions are within a few n eps of the exact one."""
    A, arrays = dense_front_problem(dominant(p + q, 1, False), p)
    fac = Plan(arrays, posdef=False).factor(A[3])
    for at in (p // 2, p - 3):
        print("case", p, q, at, flush=True)
        check(fac, arrays["perm"], True, at, p)


@pytest.mark.parametrize("s", [8, 15, 24, 32])
def test_indefinite_chains(s):
    """Fronts of s pivots and 2 s rows that form chains, one launch a band."""
    M = block_chains(s, 3)
    n = M.shape[0]
    r, c = np.nonzero(np.tril(M))
    A = g.coo_lower_to_csc(n, r, c, M[r, c])
    an = analyse(A, perm=np.arange(n), nemin=1)
    fac = Plan(an, posdef=False).factor(A[3])
    for at in (3 * s + s // 2, 9 * s + s - 2, n - 2):
        print("case chains", s, at, flush=True)
        check(fac, an.arrays()["perm"], True, at, s)


@pytest.mark.parametrize("p,q", [(20, 30), (64, 600), (100, 40), (128, 30), (200, 60)])
def test_cholesky_dense(p, q):
    """Pivots inside the 64-pivot diagonal blocks that are applied as stored
    inverses, on the vector unit (up to four right-hand sides) and on MFMA;
    condition number about 1."""
    A, arrays = dense_front_problem(dominant(p + q, 2, True), p)
    fac = Plan(arrays, posdef=True).factor(A[3])
    for at in (p // 2, p - 3):
        print("case", p, q, at, flush=True)
        check(fac, arrays["perm"], False, at, p)
