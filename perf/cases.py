"""Timed cases of the numeric phase: what a program with a fixed sparsity
pattern does once per new set of values (factor, solve, refine) or per new
right-hand side (solve), through ``opt_solver_amd.solver``.

The matrices are the library's own workloads: 7-point and 27-point SPD
operators on a cube, interior-point KKT systems on a square grid, and
trajectory-optimisation KKTs, one at a time or as a batch. The symbolic
analysis and the device plan belong to the pattern and are made once by
``prepare``, as a program that refactors would; the analysis of a pattern is
shared between preparations.

Every matrix entry and every entry of the known solution is rounded to a
power-of-two grid coarse enough that b = A x carries no rounding, in any order
of summation: x is then the exact solution, which ``exact`` returns."""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from opt_solver_amd import batch
from opt_solver_amd import generators as g
from opt_solver_amd import ordering as o
from opt_solver_amd.solver import PREC_AUTO, PREC_BF16X3, PREC_FP32, PREC_FP64, Plan, analyse

PRECISIONS = {"fp64": PREC_FP64, "fp32": PREC_FP32, "bf16x3": PREC_BF16X3, "auto": PREC_AUTO}

# kind: matrix family; size: grid side, or the longest horizon of the ocp
# systems; count: ocp systems in the batch; op: factor_solve (device-resident
# values and right-hand side), solve (a factor in hand, new right-hand sides),
# host (one call on host arrays), scaled (equilibration, scaled factor, solve,
# refinement)


def _case(name, kind, size, op="factor_solve", precision="fp64", nrhs=1, count=1):
    return {"name": name, "kind": kind, "size": size, "op": op, "precision": precision, "nrhs": nrhs,
            "count": count}


def listed():
    return [
        # one model-predictive-control step: a single short-horizon KKT from
        # host arrays in one call, where latency is all there is
        _case("mpc_step_host", "ocp", 60, op="host"),
        # a small diffusion problem refactored in a time loop
        _case("spd7_20", "spd7", 20),
        # an ordinary 3D diffusion problem, odd grid side
        _case("spd7_61", "spd7", 61),
        # an ordinary 3D elasticity-like stencil (denser rows, larger fronts)
        _case("spd27_41", "spd27", 41),
        # a large one in plain FP64
        _case("spd27_80", "spd27", 80),
        # the largest, learned mixed precision refined to FP64 accuracy
        _case("spd27_96_auto", "spd27", 96, precision="auto"),
        # many load cases against one factor
        _case("spd27_71_solve16", "spd27", 71, op="solve", nrhs=16),
        # a batch of trajectory-optimisation systems of uneven horizons
        _case("ocp_batch", "ocp", 200, count=192),
        # one iteration of a small interior-point solve, badly scaled:
        # equilibration, scaled factor, solve, refinement
        _case("kkt_70_scaled", "kkt", 70, op="scaled"),
        # an ordinary interior-point iteration in plain FP64
        _case("kkt_150", "kkt", 150),
        # a large interior-point iteration, learned mixed precision
        _case("kkt_260_auto", "kkt", 260, precision="auto"),
        # predictor and corrector right-hand sides against one KKT factor
        _case("kkt_181_solve2", "kkt", 181, op="solve", nrhs=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spd7", "spd27", "spd27", "kkt", "kkt", "ocp"])
    if kind == "ocp":
        op = rng.choice(["host", "factor_solve", "factor_solve"])
        count = 1 if op == "host" else _log_int(rng, 2, 192)
        return {"kind": kind, "size": _log_int(rng, 10, 200), "op": op, "precision": "fp64", "nrhs": 1, "count": count}
    size = _log_int(rng, 9, {"spd7": 64, "spd27": 80, "kkt": 220}[kind])
    op = rng.choice(["factor_solve", "factor_solve", "solve", "scaled" if kind == "kkt" else "host"])
    precision = rng.choice(["fp64", "auto", "bf16x3", "fp32"]) if op == "factor_solve" else "fp64"
    nrhs = rng.choice([1, 1, 2, 3, 5, 8, 13, 16]) if op in ("solve", "factor_solve") else 1
    return {"kind": kind, "size": size, "op": op, "precision": precision, "nrhs": nrhs, "count": 1}


# ---------------------------------------------------------------- patterns

@functools.lru_cache(maxsize=16)
def _spd_pattern(kind, m):
    """(n, col_ptr, row_idx, columns, Analysis) of a 7- or 27-point operator."""
    n, cp, ri, _ = g.laplace7_3d(m) if kind == "spd7" else g.spd27_3d(m, 0)
    an = analyse((n, cp, ri, None), perm=o.grid_nd((m, m, m)))
    return n, cp, ri, np.repeat(np.arange(n, dtype=np.int32), np.diff(cp)), an


def _kkt_rows(side):
    return max(1, int(round(0.32 * side * side)))


@functools.lru_cache(maxsize=16)
def _kkt_pattern(side):
    """(matrix, columns, Analysis): constraint rows join the separators of
    the grid's nested dissection."""
    m, nx = _kkt_rows(side), side * side
    A, _ = g.kkt_grid(side, m, seed=5)
    n, cp, ri, _ = A
    cols = np.repeat(np.arange(n, dtype=np.int32), np.diff(cp))
    sel = (ri >= nx) & (cols < nx)
    acols = cols[sel][np.argsort(ri[sel], kind="stable")].reshape(m, 8)
    return A, cols, analyse(A, perm=o.kkt_grid_nd(side, m, acols))


def _horizons(case):
    if case["count"] == 1:
        return [case["size"]]
    lo = max(1, min(10, case["size"]))
    return [int(t) for t in np.random.default_rng(7).integers(lo, case["size"] + 1, size=case["count"])]


@functools.lru_cache(maxsize=16)
def _ocp_pattern(horizons):
    """(arrays of the union of the systems' analyses, flops)."""
    ans = {t: analyse(g.ocp_kkt(t, seed=0), nemin=16) for t in set(horizons)}
    arrays, _ = batch.union_arrays([ans[t].arrays() for t in horizons])
    return arrays, sum(ans[t].flops for t in horizons), sum(ans[t].factor_entries for t in horizons)


# ------------------------------------------------------------------ inputs

def _grid_round(v, bits):
    return np.round(np.ldexp(v, bits)) * math.ldexp(1.0, -bits)


def _solution(case, n, seed):
    """The known solution: n x nrhs, entries in [-1, 1]."""
    bits = {"spd7": 20, "spd27": 20, "kkt": 9, "ocp": 12}[case["kind"]]
    return _grid_round(np.random.default_rng([seed, 1]).uniform(-1.0, 1.0, (case["nrhs"], n)), bits).T


def _matvec(n, cols, rows, vals, x):
    """A x of a lower matrix; every product and partial sum is exact."""
    off = rows != cols
    y = np.empty_like(x, order="F")
    for r in range(x.shape[1]):
        xr = x[:, r]
        y[:, r] = (np.bincount(rows, vals * xr[cols], n)
                   + np.bincount(cols[off], vals[off] * xr[rows[off]], n))
    return y


def _matrix(case, seed):
    """(analysis for Plan, n, columns, rows, values) of the seed's matrix."""
    rng = np.random.default_rng([seed, 0])
    if case["kind"] in ("spd7", "spd27"):
        # variable-coefficient operator, strictly diagonally dominant
        n, cp, ri, cols, an = _spd_pattern(case["kind"], case["size"])
        vals = -_grid_round(rng.uniform(0.5, 1.5, ri.size), 20)
        first = cp[:-1]
        vals[first] = 0.0
        vals[first] = -(np.bincount(ri, vals, n) + np.bincount(cols, vals, n)) + 2.0**-10
        return an, n, cols, ri, vals
    if case["kind"] == "kkt":
        # a later interior-point iterate: every barrier weight moved on its
        # own, the constraint Jacobian unchanged
        A, cols, an = _kkt_pattern(case["size"])
        nx = case["size"] ** 2
        vals = _grid_round(A[3], 16)
        first = A[1][:-1]
        vals[first[:nx]] = 4.0 + _grid_round(10.0 ** rng.uniform(-6.0, 6.0, nx), 22)
        vals[first[nx:]] = -(2.0**-27)
        return an, A[0], cols, A[2], vals
    horizons = _horizons(case)
    arrays, _, _ = _ocp_pattern(tuple(horizons))
    mats = [g.ocp_kkt(t, seed=int(s)) for t, s in zip(horizons, rng.integers(1 << 30, size=len(horizons)))]
    start = np.cumsum([0] + [M[0] for M in mats])
    cols = np.concatenate([np.repeat(np.arange(M[0]), np.diff(M[1])) + b for M, b in zip(mats, start)])
    rows = np.concatenate([M[2] + b for M, b in zip(mats, start)])
    return arrays, int(start[-1]), cols, rows, _grid_round(np.concatenate([M[3] for M in mats]), 30)


def prepare(case, seed):
    an, n, cols, rows, vals = _matrix(case, seed)
    b = _matvec(n, cols, rows, vals, _solution(case, n, seed))
    plan = Plan(an, posdef=case["kind"] in ("spd7", "spd27"))
    state = {"case": case, "plan": plan}
    if case["op"] == "host":
        return {**state, "vals": vals, "b": b[:, 0]}
    state["vals"] = torch.from_numpy(np.ascontiguousarray(vals)).cuda()
    state["b"] = torch.from_numpy(np.ascontiguousarray(b.T)).cuda()  # nrhs x n: each system contiguous
    state["x"] = torch.empty_like(state["b"])
    torch.cuda.synchronize()
    if case["op"] == "solve":
        state["factor"] = plan.factor(values_ptr=state["vals"].data_ptr())
    return state


# --------------------------------------------------------------------- run

def _counts(fac):
    return np.array([*fac.inertia, fac.info.delayed_pivots, fac.info.two_by_two_pivots], dtype=np.int64)


def run(state):
    case, plan, b = state["case"], state["plan"], state["b"]
    if case["op"] == "host":
        fac, x, _ = plan.factor_solve(state["vals"], b)
        return {"x": x, "counts": _counts(fac)}
    vp, x = state["vals"].data_ptr(), state["x"]
    if case["op"] == "solve":
        fac = state["factor"]
    elif case["op"] == "scaled":
        fac = plan.factor(values_ptr=vp, scale=plan.equilibration_scale(values_ptr=vp))
    else:
        fac = plan.factor(values_ptr=vp, precision=PRECISIONS[case["precision"]])
    x.copy_(b)
    torch.cuda.current_stream().synchronize()  # the library works on a stream of its own
    fac.solve_device(x.data_ptr(), case["nrhs"])
    if case["op"] == "scaled" or case["precision"] != "fp64":
        fac.refine_device(b.data_ptr(), x.data_ptr(), case["nrhs"])
    return {"x": x, "counts": _counts(fac)}


# -------------------------------------------------------------------- work

def _sizes(case):
    """(n, entries, flops, factor entries)."""
    if case["kind"] in ("spd7", "spd27"):
        n, _, ri, _, an = _spd_pattern(case["kind"], case["size"])
        return n, ri.size, an.flops, an.factor_entries
    if case["kind"] == "kkt":
        A, _, an = _kkt_pattern(case["size"])
        return A[0], A[2].size, an.flops, an.factor_entries
    arrays, flops, entries = _ocp_pattern(tuple(_horizons(case)))
    return int(arrays["n"]), int(arrays["orig_to_slot"].size), flops, entries


def work(case):
    n, nnz, flops, entries = _sizes(case)
    rhs = case["nrhs"]
    sweeps = 4.0 * entries * rhs  # a multiply and an add per factor entry, forward and backward
    if case["op"] == "solve":  # the factor and b read, x written
        return {"bytes": 8 * entries + 16 * n * rhs, "flops": sweeps}
    # values and b read, the factor (kept for later solves) and x written
    return {"bytes": 8 * (nnz + entries) + 16 * n * rhs, "flops": flops + sweeps}


# ------------------------------------------------------------------- exact

def _inertia(case, n):
    """Positive, negative and zero eigenvalues of the family's matrices."""
    if case["kind"] == "kkt":
        neg = _kkt_rows(case["size"])
    else:
        neg = 12 * sum(_horizons(case)) if case["kind"] == "ocp" else 0
    return n - neg, neg, 0


def _order(case):
    if case["kind"] in ("spd7", "spd27"):
        return case["size"] ** 3
    if case["kind"] == "kkt":
        return case["size"] ** 2 + _kkt_rows(case["size"])
    return sum(28 * t + 12 for t in _horizons(case))


def exact(case, seed):
    x = _solution(case, _order(case), seed)
    x = x[:, 0] if case["op"] == "host" else np.ascontiguousarray(x.T)
    return {"x": x, "counts": None}
