"""Kernels at the sizes where their tiles and remainders begin and end,
against the oracle's factor of the same analysis and known solutions."""
import numpy as np
import pytest

from tests.conftest import gpu_available
from tests.helpers import dense_front_problem, matvec

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no GPU", allow_module_level=True)

from opt_solver_amd import generators as g  # noqa: E402
from opt_solver_amd._lib import TUNE_SOLVE_FUSE_ROWS  # noqa: E402
from opt_solver_amd.solver import Plan, analyse  # noqa: E402
from tests.test_gpu_spd import block_rel_err  # noqa: E402


def dense_spd(n, seed):
    """A dense symmetric positive definite matrix (one supernode): G G^T / n
    + I has a condition number of about 5."""
    rng = np.random.default_rng([n, seed])
    G = rng.standard_normal((n, n))
    M = G @ G.T / n + np.eye(n)
    r, c = np.tril_indices(n)
    return g.coo_lower_to_csc(n, r, c, M[r, c])


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 47, 48, 49, 63, 64, 65, 81, 128, 129, 200])
def test_dense_cholesky_panel_edges(oracle_lib, n):
    """One front of n pivots: diagonal blocks of every remainder modulo 16
    and 64. Both factors are within n eps cond (200 x 2.2e-16 x 5 = 2e-13)
    of the exact one."""
    print("case dense", n, flush=True)
    A = dense_spd(n, 1)
    an = analyse(A)
    assert an.nsup == 1
    fac = Plan(an, posdef=True).factor(A[3])
    orc = oracle_lib.Factor(an.arrays(), A[3], posdef=True)
    assert fac.status == 0
    assert block_rel_err(fac.export(), orc.export()) < 4e-13
    x = np.random.default_rng(n).uniform(-1, 1, n)
    assert np.abs(fac.solve(matvec(A, x)) - x).max() < 1e-12


@pytest.mark.parametrize("n,bad", [(1, 0), (16, 15), (40, 16), (64, 63), (70, 65)])
def test_dense_cholesky_bad_pivot(n, bad):
    """A pivot that is zero or negative at the edge of a panel is reported."""
    for shift in (0.0, -1.0):
        n_, cp, ri, v = dense_spd(n, 2)
        M = g.csc_to_dense(n, cp, ri, v)
        L = np.linalg.cholesky(M)
        v = v.copy()
        v[cp[bad]] += shift * 1e-3 - L[bad, bad] ** 2 * (1.0 if shift else 1.0 + 1e-9)
        fac = Plan(analyse((n, cp, ri, v)), posdef=True).factor(v)
        assert fac.status == 1


@pytest.mark.parametrize("p,q", [(1, 0), (63, 65), (64, 512), (64, 513), (65, 1), (128, 64), (129, 700), (191, 3),
                                 (192, 0), (193, 40), (255, 600), (256, 1), (257, 512), (320, 0), (513, 65)])
def test_indefinite_sweep_edges(p, q):
    """Sweeps of an LDL^T factor whose first front has p pivots and q rows
    below them (a dense front of p + q rows split in two supernodes):
    sub-blocks of 64, steps of 256, the fused limits of 64 pivots and 512
    rows, every number of right-hand sides a pass holds. The matrix is a
    random symmetric one plus an alternating diagonal of +-2 n, so its
    solution is known to about n eps."""
    n = p + q
    print("case sweep", p, q, flush=True)
    rng = np.random.default_rng([p, q])
    M = rng.uniform(-1, 1, (n, n))
    M = M + M.T + np.diag(2.0 * n * np.where(np.arange(n) % 3 == 0, -1.0, 1.0))
    A, arrays = dense_front_problem(M, p)
    fac = Plan(arrays, posdef=False).factor(A[3])
    assert fac.status == 0
    X = rng.uniform(-1, 1, (n, 7))
    B = M @ X
    for nr in (1, 2, 3, 7):
        xs = fac.solve(B[:, :nr] if nr > 1 else B[:, 0]).reshape(n, nr)
        assert np.abs(xs - X[:, :nr]).max() < 1e-13 * max(n, 10)


@pytest.mark.parametrize("p,q", [(1, 0), (1, 1), (3, 1), (63, 66), (64, 511), (64, 513), (65, 2), (127, 129),
                                 (128, 0), (129, 640), (191, 1), (192, 257), (193, 256), (256, 255), (320, 1100)])
def test_cholesky_sweep_edges(p, q):
    """Sweeps of a Cholesky factor whose first front has p pivots and q rows
    below them: 64-pivot blocks, 128-pivot steps, 64- and 128-row groups,
    odd row counts (pairs of rows), 256-row stages, 512-row segments, and 1,
    4, 16 and more right-hand sides. Condition number about 5."""
    n = p + q
    print("case cholesky sweep", p, q, flush=True)
    rng = np.random.default_rng([p, q, 1])
    G = rng.standard_normal((n, n))
    M = G @ G.T / n + np.eye(n)
    A, arrays = dense_front_problem(M, p)
    plan = Plan(arrays, posdef=True)
    fac = plan.factor(A[3])
    assert fac.status == 0
    X = rng.uniform(-1, 1, (n, 18))
    B = M @ X
    for fuse in (512, 0, 1 << 20):
        plan.tune(TUNE_SOLVE_FUSE_ROWS, fuse)
        for nr in (1, 3, 4, 5, 16, 18):
            xs = fac.solve(B[:, :nr] if nr > 1 else B[:, 0]).reshape(n, nr)
            assert np.abs(xs - X[:, :nr]).max() < 1e-14 * max(n, 100), (fuse, nr)


def block_chains(s, seed):
    """Blocks of s columns: a chain of seven, then two chains of four and
    two that meet in a third of three. Dense blocks on the diagonal and
    between neighbours, diagonal of alternating sign twice the row sums."""
    links = [(i, i + 1) for i in range(6)] + [(7, 8), (8, 9), (9, 10), (10, 13), (11, 12), (12, 13), (13, 14), (14, 15)]
    nb, rng = 16, np.random.default_rng([s, seed])
    M = np.zeros((nb * s, nb * s))
    for i, j in links + [(i, i) for i in range(nb)]:
        M[j * s:(j + 1) * s, i * s:(i + 1) * s] = rng.uniform(0.1, 1, (s, s))
    M = np.tril(M, -1)
    M = M + M.T
    n = nb * s
    return M + np.diag(np.where(np.arange(n) % 3 == 0, -2.0, 2.0) * (M.sum(1) + 1.0))


@pytest.mark.parametrize("s", [1, 2, 8, 15, 16, 17, 24, 31, 32, 33])
def test_chain_bands(s):
    """Chains of fronts of 2 s rows: one launch a band while the rows are at
    most 64, columns in groups of 16 with 32 read ahead, one wavefront up to
    48 rows and a workgroup above, chains of one front and more, every number
    of right-hand sides a pass holds. Strictly diagonally dominant by a factor
    of two: the solution is known to a few n eps."""
    print("case chains", s, flush=True)
    M = block_chains(s, 0)
    n = M.shape[0]
    r, c = np.nonzero(np.tril(M))
    A = g.coo_lower_to_csc(n, r, c, M[r, c])
    fac = Plan(analyse(A, perm=np.arange(n), nemin=1), posdef=False).factor(A[3])
    assert fac.status == 0
    X = np.random.default_rng(s).uniform(-1, 1, (n, 18))
    B = M @ X
    for nr in (1, 2, 3, 16, 18):
        xs = fac.solve(B[:, :nr] if nr > 1 else B[:, 0]).reshape(n, nr)
        assert np.abs(xs - X[:, :nr]).max() < 1e-13 * max(n, 10), nr


@pytest.mark.parametrize("delayed", [False, True])
@pytest.mark.parametrize("p,q", [(1, 96), (3, 1021), (3, 1024), (3, 1025), (2, 2047), (3, 2049), (70, 960)])
def test_indefinite_assembly_edges(p, q, delayed):
    """A root of q rows (p more with the child's delayed columns) assembled
    from one child: a wavefront per column up to 1024 rows, a workgroup with
    2048-row chunks above, groups of 8 columns, and the root's updates in 64 x
    64 tiles. delayed: the child's block is zero, so all its columns reach the
    root; the matrix is then [0 B; B^T D] with D = 2 n I, B uniform in [-1,
    1], of condition number about 12 n, solved to well below 1e-13 n."""
    n = p + q
    print("case assembly", p, q, delayed, flush=True)
    rng = np.random.default_rng([p, q, 3])
    M = rng.uniform(-1, 1, (n, n))
    M = M + M.T
    d = np.full(n, 2.0 * n) if delayed else 2.0 * n * np.where(np.arange(n) % 3 == 0, -1.0, 1.0)
    M += np.diag(d)
    if delayed:
        M[:p, :p] = 0.0
        M[p:, p:] = np.diag(d[p:])
    A, arrays = dense_front_problem(M, p)
    fac = Plan(arrays, posdef=False).factor(A[3])
    assert fac.status == 0
    neg = p if delayed else int((d < 0).sum())
    assert fac.inertia == (n - neg, neg, 0)
    x = rng.uniform(-1, 1, n)
    assert np.abs(fac.solve(M @ x) - x).max() < 1e-13 * max(n, 10)


@pytest.mark.parametrize("p,q", [(17, 100), (18, 78), (20, 201), (32, 300)])
def test_panel_stalls_with_no_live_column_left(oracle_lib, p, q):
    """A first front of p eligible columns, none of which is an acceptable
    pivot (entries of 1 between them, of 1e6 below them): its first panel
    stalls, pulls the partners from behind it, stalls at the same position and
    is rotated away, and what was pulled stalls there again as the last live
    columns, with nothing to exchange. Counters, delays and inertia are the
    oracle's."""
    n = p + q
    print("case last live columns", p, q, flush=True)
    rng = np.random.default_rng([p, q, 5])
    M = np.zeros((n, n))
    for j in range(16, p):
        M[j, j - 16] = 1.0
    M[p:, :p] = 1e6 * rng.uniform(0.5, 1, (q, p))
    M = M + M.T
    M[p:, p:] = np.diag(2e6 * n * np.where(np.arange(q) % 3 == 0, -1.0, 1.0))
    A, arrays = dense_front_problem(M, p)
    fac = Plan(arrays, posdef=False).factor(A[3])
    orc = oracle_lib.Factor(arrays, A[3], posdef=False)
    front = oracle_lib.ldlt_front(M, p)[3]
    assert (front["stalls"], front["pulls"], front["rotated"]) == (3, min(p - 16, 8), p), front  # 16 / 2 pairs at most
    assert fac.status == orc.status == 0 and fac.inertia == orc.inertia
    assert tuple(fac.stall_stats()[0]) == (front["stalls"], front["pulls"], front["rotated"], front["searches"])
    assert fac.info.delayed_pivots == orc.delayed == p
    x = rng.uniform(-1, 1, n)
    eta, _ = oracle_lib.backward_error(A, M @ x, fac.solve(M @ x))
    assert eta < 1e-13  # n eps


@pytest.mark.parametrize("prec", ["bf16x3", "bf16"])
def test_odd_fronts_on_planes_bitwise(prec):
    """Several large fronts of odd row and column counts below 1024 in one
    level, so that no front's operand planes have a round length: the same
    factor, bit for bit, as with the operands rounded inside every tile."""
    from opt_solver_amd import batch
    from opt_solver_amd._lib import TUNE_LDLT_OUTER_WIDE, TUNE_LDLT_PLANES
    from opt_solver_amd.solver import PREC_BF16, PREC_BF16X3
    print("case odd planes", prec, flush=True)
    rng = np.random.default_rng(11)
    systems, vals = [], []
    for f, ne in ((901, 301), (1301, 901), (777, 535), (1175, 1023)):
        M = rng.uniform(-1, 1, (f, f))
        M = M + M.T + np.diag(4.0 * f * np.where(np.arange(f) % 3 == 0, -1.0, 1.0))
        A, arrays = dense_front_problem(M, ne)
        systems.append(arrays)
        vals.append(A[3])
    plan = Plan(batch.union_arrays(systems)[0], posdef=False)
    plan.tune(TUNE_LDLT_OUTER_WIDE, 512)
    ex = []
    for planes in (1, 0):
        plan.tune(TUNE_LDLT_PLANES, planes)
        fac = plan.factor(np.concatenate(vals), precision={"bf16x3": PREC_BF16X3, "bf16": PREC_BF16}[prec],
                          mixed_min_front=512)
        assert fac.status == 0 and fac.info.fronts_reduced >= 4
        ex.append(fac.export())
    for key in ("steps", "row_indices", "pivot_types", "factor_values"):
        assert np.array_equal(ex[0][key], ex[1][key]), key


@pytest.mark.parametrize("ne,f", [(60, 96), (150, 200), (100, 255), (100, 256), (200, 300)])
def test_reduced_precision_starts_at_256_rows(ne, f):
    """An indefinite factorization below FP64 keeps fronts of fewer than 256
    rows in FP64 whatever mixed_min_front says, and takes no training pair
    from them, unless the plan's large-front line is set lower."""
    from opt_solver_amd._lib import TUNE_LDLT_BIG_MIN
    from opt_solver_amd.solver import PREC_FP32, PREC_FP64
    print("case reduced", ne, f, flush=True)
    rng = np.random.default_rng([ne, f])
    M = rng.uniform(-1, 1, (f, f))
    M = M + M.T + np.diag(4.0 * f * np.where(np.arange(f) % 3 == 0, -1.0, 1.0))
    A, arrays = dense_front_problem(M, ne)
    plan = Plan(arrays, posdef=False)
    want = 1 if f >= 256 else 0
    fac = plan.factor(A[3], precision=PREC_FP32, mixed_min_front=64)
    # (the root has f - ne < 256 rows)
    assert fac.info.fronts_reduced == want and (fac.precisions()[0] != PREC_FP64) == bool(want)
    if not want:
        low = fac.export()["factor_values"]
        assert np.array_equal(low, plan.factor(A[3]).export()["factor_values"])
    fac = plan.factor(A[3], collect=True, mixed_min_front=64)
    assert list(fac.selector_pairs()[2]) == [0] * want
    plan.tune(TUNE_LDLT_BIG_MIN, 96)
    assert plan.factor(A[3], precision=PREC_FP32, mixed_min_front=64).precisions()[0] == PREC_FP32


@pytest.mark.parametrize("panel,wide", [(511, 1024), (513, 1024), (700, 1024), (2000, 1024), (2**31 - 1, 1024), (100, 64)])
def test_panels_wider_than_the_outer_block(panel, wide):
    """Panel widths up to and past the large fronts' outer block of 512
    columns (and past its workspace), or of 64 where the plan's planes are
    tuned to it: the solution is known to about n eps."""
    from opt_solver_amd._lib import TUNE_LDLT_OUTER_WIDE
    from opt_solver_amd.solver import PREC_BF16X3, PREC_FP64
    print("case panel", panel, wide, flush=True)
    ne, n = 1300, 1400
    rng = np.random.default_rng(panel % 1000)
    M = rng.uniform(-1, 1, (n, n))
    M = M + M.T + np.diag(4.0 * n * np.where(np.arange(n) % 3 == 0, -1.0, 1.0))
    A, arrays = dense_front_problem(M, ne)
    plan = Plan(arrays, posdef=False)
    plan.tune(TUNE_LDLT_OUTER_WIDE, wide)
    x = rng.uniform(-1, 1, n)
    fac = plan.factor(A[3], panel=panel)
    assert fac.status == 0 and fac.inertia == (n - (n + 2) // 3, (n + 2) // 3, 0)
    assert np.abs(fac.solve(M @ x) - x).max() < 1e-13 * n
    # split BF16 products are within 2^-16 of the entries', which are at most
    # 1 / (2 n) of the diagonal
    fac = plan.factor(A[3], panel=panel, precision=PREC_BF16X3, mixed_min_front=1024)
    assert fac.precisions()[0] != PREC_FP64
    assert np.abs(fac.solve(M @ x) - x).max() < 1e-6
