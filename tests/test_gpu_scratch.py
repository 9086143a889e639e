"""Device memory that a plan's calls take, as its statistics report it."""
import numpy as np
import pytest

from tests.conftest import gpu_available
from tests.helpers import dense_front_problem, matvec

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no GPU", allow_module_level=True)

import torch  # noqa: E402

from opt_solver_amd import batch  # noqa: E402
from opt_solver_amd import generators as g  # noqa: E402
from opt_solver_amd.solver import Plan, analyse  # noqa: E402


def many_fronts(count, f):
    """(growth of the plan's device memory by a factorization, error of the
    solutions) of `count` dense systems of f rows in one level: alternating
    diagonal of 2 f, entries in [-1, 1], system k scaled by 2^(k mod 8)."""
    rng = np.random.default_rng(f)
    M = rng.uniform(-1, 1, (f, f))
    M = M + M.T + np.diag(4.0 * f * np.where(np.arange(f) % 3 == 0, -1.0, 1.0))
    A, arrays = dense_front_problem(M, f)
    union, _ = batch.union_arrays([arrays] * count)
    scale = 2.0 ** (np.arange(count) % 8)
    plan = Plan(union, posdef=False)
    vals = torch.from_numpy((scale[:, None] * A[3]).reshape(-1)).cuda()
    X = rng.uniform(-1, 1, (count, f))
    b = torch.from_numpy((scale[:, None] * (X @ M)).reshape(-1)).cuda()
    torch.cuda.synchronize()
    before = plan.stats()["device_bytes"]
    fac = plan.factor(values_ptr=vals.data_ptr())
    after = plan.stats()["device_bytes"]
    assert fac.status == 0 and fac.inertia[1] == count * -(-f // 3)
    fac.solve_device(b.data_ptr(), 1)
    return after - before, np.abs(b.cpu().numpy().reshape(count, f) - X).max()


@pytest.mark.parametrize("f,count", [(96, 7000), (131, 5000)])
def test_level_of_many_large_fronts(f, count):
    """The working memory of a level's large fronts (96 rows and more) does
    not grow with their number: a panel workspace and a group buffer are 187
    KB a front at 96 rows and 278 KB at 131, all of these together 1.3 GB, of
    which a factorization takes 1 GiB at most, and below 4 KB a front for
    records and lists. The solutions are known to about f eps."""
    print("case", count, "fronts of", f, flush=True)
    grown, err = many_fronts(count, f)
    print("grown", grown, flush=True)
    assert err < 1e-13 * f
    assert grown < 2**30 + 4096 * count


def test_solve_buffer_settles_at_the_first_call():
    """A plan's right-hand-side block is sized by its first solve: no later
    call with more right-hand sides frees and allocates it again."""
    for posdef in (True, False):
        A = g.laplace7_3d(9)
        plan = Plan(analyse(A), posdef=posdef)
        fac = plan.factor(A[3])
        X = np.random.default_rng(3).uniform(-1, 1, (A[0], 33))
        B = torch.from_numpy(np.ascontiguousarray(matvec(A, X).T)).cuda()
        sizes = []
        for nr in (1, 2, 5, 16, 33):
            x = B[:nr].clone()
            torch.cuda.synchronize()
            fac.solve_device(x.data_ptr(), nr)
            assert np.abs(x.cpu().numpy().T - X[:, :nr]).max() < 1e-11
            sizes.append(plan.stats()["device_bytes"])
        assert len(set(sizes)) == 1, (posdef, sizes)
