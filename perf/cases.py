"""Performance cases of the numeric phase: what a program that uses the solver has it do.

Every case is a refactorization, a solve, or both, of one analyzed pattern through the public interface (the
C-ABI of include/symla_hip.h, or the SymLDLT class for host arrays).  ``listed`` names the representative ones,
``draw`` gives more of the same ranges.

The matrices are the ones of the benchmark configurations and tests (grid Laplacians with variable coefficients,
the 27-point stencil, SQD KKT systems, batches of small 2D systems), shifted to be indefinite.  Their entries and
the solutions are rounded to a fixed number of binary places, so that B = A X is formed without any rounding and
the X the inputs are made from is the exact solution of the system.
"""
from __future__ import annotations

import ctypes as C
import functools

import numpy as np
import torch

from ma57_amd import _lib, problems
from ma57_amd.solver import Mode, OrderingType, Precision, SymLDLT

PRECISIONS = {"fp64": Precision.FP64, "fp32": Precision.FP32, "bf16x3": Precision.BF16X3}
REFINE_ITERATIONS, REFINE_TOLERANCE = 10, 1e-12
X_STEP, A_STEP = 2.0 ** -16, 2.0 ** -20


def listed():
    return [
        # the smallest call: host arrays in and out, one right-hand side (an optimizer's or a test's small system)
        dict(name="grid2d_24_host", kind="grid2d", dims="24x24", shift=0.3, ordering="amd", op="host",
             precision="fp64", refine=False, nrhs=1),
        # a 2D mesh refactored and solved once per time step
        dict(name="grid2d_100", kind="grid2d", dims="100x100", shift=0.3, ordering="amd", op="factor_solve",
             precision="fp64", refine=False, nrhs=1),
        # a 3D mesh with a few load cases
        dict(name="grid3d_40", kind="grid3d", dims="40x40x40", shift=0.5, ordering="nd", op="factor_solve",
             precision="fp64", refine=False, nrhs=16),
        # the same on an uneven box in mixed precision: FP32 fronts, FP64 refinement
        dict(name="grid3d_37x41x43_fp32", kind="grid3d", dims="37x41x43", shift=0.5, ordering="nd",
             op="factor_solve", precision="fp32", refine=True, nrhs=5),
        # new right-hand side on an existing factorization, one at a time (a time loop with a fixed matrix)
        dict(name="grid3d_40_solve1", kind="grid3d", dims="40x40x40", shift=0.5, ordering="nd", op="solve",
             precision="fp64", refine=False, nrhs=1),
        # an interior-point step: static-regularized KKT factorization with inertia control, refined solve
        dict(name="kkt_30_static", kind="kkt", dims="30", shift=0.0, ordering="amd", op="factor_solve",
             precision="fp64", refine=True, nrhs=4),
        # many independent small systems in one plan
        dict(name="batch_192", kind="batch", dims="192", shift=0.0, ordering="amd", op="factor_solve",
             precision="fp64", refine=False, nrhs=1),
        # a recorded refactorize + refined solve, replayed on new values (a Newton loop)
        dict(name="stencil27_30_graph", kind="stencil27", dims="30x30x30", shift=0.2, ordering="nd", op="graph",
             precision="fp32", refine=True, nrhs=64),
        # many right-hand sides on an existing factorization
        dict(name="stencil27_40_solve64", kind="stencil27", dims="40x40x40", shift=0.2, ordering="nd", op="solve",
             precision="fp64", refine=False, nrhs=64),
        # a large 3D problem in plain FP64
        dict(name="stencil27_64", kind="stencil27", dims="64x64x64", shift=0.2, ordering="nd", op="factor_solve",
             precision="fp64", refine=False, nrhs=64),
        # an uneven one with split-BF16 contribution-block updates
        dict(name="stencil27_53x57x59_bf16x3", kind="stencil27", dims="53x57x59", shift=0.2, ordering="nd",
             op="factor_solve", precision="bf16x3", refine=True, nrhs=33),
        # the benchmark's own workload: the largest, FP32 fronts with FP64 refinement
        dict(name="stencil27_80_fp32", kind="stencil27", dims="80x80x80", shift=0.2, ordering="nd",
             op="factor_solve", precision="fp32", refine=True, nrhs=64),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """One more case: every kind of system and call, sizes over the whole range (odd ones included)."""
    kind = rng.choice(["grid2d", "grid2d", "grid3d", "grid3d", "stencil27", "stencil27", "kkt", "batch"])
    precision = rng.choice(["fp64", "fp64", "fp32"])
    op = rng.choice(["factor_solve", "factor_solve", "solve", "graph"])
    ordering = "nd"
    shift = 0.0
    nrhs = _log_int(rng, 1, 64)
    if kind == "grid2d":
        dims = [_log_int(rng, 12, 320) for _ in range(2)]
        ordering, shift = rng.choice(["amd", "nd"]), 0.3
        if dims[0] * dims[1] <= 10000 and op == "factor_solve":
            op = rng.choice(["host", "factor_solve"])
    elif kind == "grid3d":
        dims, shift = [_log_int(rng, 8, 48) for _ in range(3)], 0.5
    elif kind == "stencil27":
        dims, shift = [_log_int(rng, 8, 56) for _ in range(3)], 0.2
        if precision == "fp32" and rng.random() < 0.4:
            precision = "bf16x3"
    elif kind == "kkt":
        dims, ordering, op = [_log_int(rng, 8, 26)], "amd", "factor_solve"
        nrhs = min(nrhs, 16)
    else:
        dims, ordering, op = [_log_int(rng, 3, 256)], "amd", "factor_solve"
        nrhs = min(nrhs, 8)
    refine = precision != "fp64" or kind == "kkt" or rng.random() < 0.2
    if op == "host":
        precision, refine = "fp64", False
    return dict(kind=kind, dims="x".join(map(str, dims)), shift=shift, ordering=ordering, op=op, precision=precision,
                refine=refine, nrhs=nrhs)


# --- systems -------------------------------------------------------------------------------------------------

def _grid(dims, stencil27):
    """Lower-triangle CSC pattern (colptr, row, col) of a grid with 2 neighbours per axis, or all 3^d - 1."""
    nd = len(dims)
    coords = np.meshgrid(*[np.arange(k) for k in dims], indexing="ij")
    strides = [int(np.prod(dims[a + 1:])) for a in range(nd)]
    offs = [o for o in np.ndindex(*([3] * nd)) if o >= (1,) * nd]
    offs = [tuple(v - 1 for v in o) for o in offs]
    if not stencil27:
        offs = [o for o in offs if sum(map(abs, o)) <= 1]
    offs.sort(key=lambda o: sum(v * s for v, s in zip(o, strides)))
    n = int(np.prod(dims))
    ok = np.empty((n, len(offs)), bool)
    for k, o in enumerate(offs):
        m = np.ones(dims, bool)
        for a in range(nd):
            m &= (coords[a] + o[a] >= 0) & (coords[a] + o[a] < dims[a])
        ok[:, k] = m.ravel()
    delta = np.array([sum(v * s for v, s in zip(o, strides)) for o in offs], np.int64)
    rows = np.arange(n)[:, None] + delta[None, :]
    colptr = np.concatenate([[0], np.cumsum(ok.sum(axis=1))]).astype(np.int64)
    row = rows[ok].astype(np.int32)
    return n, colptr, row, np.repeat(np.arange(n, dtype=np.int32), np.diff(colptr))


def _round(v, step):
    return np.round(v / step) * step


def _patterns(case):
    """[(n, colptr, row, col, base values or None)]: one pattern per independent system of the case."""
    dims = [int(k) for k in case["dims"].split("x")]
    if case["kind"] in ("grid2d", "grid3d", "stencil27"):
        return [_grid(dims, case["kind"] == "stencil27") + (None,)]
    if case["kind"] == "kkt":
        systems = [problems.sqd_kkt(dims[0], dims[0] ** 3 // 3)[0]]
    else:
        systems = [problems.batched_system(problems.SEED_BASE + 4 + 1000 * i) for i in range(dims[0])]
    out = []
    for A in systems:
        cp = A.indptr.astype(np.int64)
        out.append((A.shape[0], cp, A.indices.astype(np.int32),
                    np.repeat(np.arange(A.shape[0], dtype=np.int32), np.diff(cp)), A.data))
    return out


def _values(case, pattern, rng):
    n, cp, row, col, base = pattern
    if case["kind"] == "batch":  # the system's coefficients, a few per cent apart
        return _round(base * rng.uniform(0.95, 1.05, base.size), A_STEP)
    if case["kind"] == "kkt":  # [[-(H + eps_h I), J^T], [J, eps_f I]] with a new J
        n1 = int(case["dims"]) ** 3
        vals = np.round(base)
        j = (row >= n1) & (col < n1)
        vals[j] = _round(rng.standard_normal(int(j.sum())), X_STEP) + X_STEP
        d = row == col
        vals[d & (row < n1)] -= 2.0 ** -13
        vals[d & (row >= n1)] = 2.0 ** -27
        return vals
    # -w per edge, w ~ U(0.5, 1.5); the diagonal is the sum over all neighbours (1 for those outside), less the shift
    off = row != col
    w = _round(rng.uniform(0.5, 1.5, int(off.sum())), A_STEP)
    full = {"grid2d": 4, "grid3d": 6, "stencil27": 26}[case["kind"]]
    diag = np.zeros(n)
    deg = np.zeros(n)
    for end in (row[off], col[off]):
        diag += np.bincount(end, weights=w, minlength=n)
        deg += np.bincount(end, minlength=n)
    vals = np.empty(row.size)
    vals[off] = -w
    vals[~off] = diag + (full - deg) - _round(np.float64(case["shift"]), A_STEP)
    return vals


def _order(case):
    n_all = [p[0] for p in _patterns_cached(_key(case))]
    return n_all, int(sum(n_all))


def _key(case):
    return (case["kind"], case["dims"])


@functools.lru_cache(maxsize=1)
def _patterns_cached(key):
    return _patterns({"kind": key[0], "dims": key[1]})


def _solution(n, nrhs, seed):
    rng = torch.Generator().manual_seed(seed * 1000003 + 17)
    x = torch.randn((nrhs, n), dtype=torch.float32, generator=rng).double()
    return torch.round(x / X_STEP) * X_STEP


def _product(n, row, col, vals, x):
    """A x for every row of x, A symmetric from its lower triangle (every sum is exact, whatever its order)."""
    r, c, v = (torch.as_tensor(a).to(x.device) for a in (row.astype(np.int64), col.astype(np.int64), vals))
    off = r != c
    b = torch.empty_like(x)
    for k in range(x.shape[0]):
        y = torch.zeros(n, dtype=x.dtype, device=x.device)
        y.index_add_(0, r, v * x[k][c])
        y.index_add_(0, c[off], v[off] * x[k][r[off]])
        b[k] = y
    return b


# --- the calls -----------------------------------------------------------------------------------------------

def _ptr(t):
    return C.c_void_p(t.data_ptr())


class _System:
    """An analyzed pattern and its plan, through the C-ABI."""

    def __init__(self, patterns, ordering):
        self.lib = _lib.load()
        self.sym, self.plan = C.c_void_p(), C.c_void_p()
        order = _lib.ORDER_AMD if ordering == "amd" else _lib.ORDER_METIS
        self.sizes = np.array([p[0] for p in patterns], np.int32)
        self.starts = np.concatenate([[0], np.cumsum(self.sizes)]).astype(np.int32)
        self.n = int(self.starts[-1])
        ns = len(patterns)
        if ns == 1:
            n, cp, row = patterns[0][:3]
            args = (_lib.ptr(cp, _lib.i64p), _lib.ptr(row, _lib.i32p))
            self._ok(self.lib.symla_analyze(n, *args, order, None, 64, 0.25, C.byref(self.sym)))
            self.make = lambda out: self.lib.symla_plan_create(self.sym, *args, out)
        else:
            cps = (_lib.i64p * ns)(*[_lib.ptr(p[1], _lib.i64p) for p in patterns])
            rows = (_lib.i32p * ns)(*[_lib.ptr(p[2], _lib.i32p) for p in patterns])
            sizes = _lib.ptr(self.sizes, _lib.i32p)
            self._ok(self.lib.symla_batch_analyze(ns, sizes, cps, rows, order, 64, 0.25, C.byref(self.sym)))
            self.make = lambda out: self.lib.symla_batch_plan_create(self.sym, ns, sizes, cps, rows, out)

    def create(self):
        self._ok(self.make(C.byref(self.plan)))

    def _ok(self, rc):
        if rc:
            msg = self.lib.symla_plan_last_error(self.plan) if self.plan else self.lib.symla_last_error()
            raise RuntimeError(msg.decode())

    def options(self, precision, signs=None):
        o = _lib.FactorOpts()
        o.mode = Mode.ThresholdPivot if signs is None else Mode.StaticRegularized
        o.pivot_threshold, o.zero_tolerance, o.relative_pivot_floor = 0.01, 1e-300, 1e-12
        o.expected_sign = _lib.ptr(signs, _lib.i32p) if signs is not None else None
        o.initial_delta, o.max_retries, o.growth = 0.0, 10, 10.0
        o.static_rel_floor, o.static_abs_floor = 1e-8, 1e-300
        o.precision = precision
        return o

    def __del__(self):
        if self.plan:
            self.lib.symla_plan_destroy(self.plan)
        if self.sym:
            self.lib.symla_symbolic_free(self.sym)


def prepare(case, seed):
    patterns = _patterns_cached(_key(case))
    rng = np.random.default_rng(seed * 7919 + 11)
    per = [_values(case, p, rng) for p in patterns]
    starts = np.concatenate([[0], np.cumsum([p[0] for p in patterns])])
    n, nrhs = int(starts[-1]), case["nrhs"]
    x = _solution(n, nrhs, seed).cuda()
    rows = np.concatenate([p[2].astype(np.int64) + s for p, s in zip(patterns, starts)])
    cols = np.concatenate([p[3].astype(np.int64) + s for p, s in zip(patterns, starts)])
    vals = np.concatenate(per)
    b = _product(n, rows, cols, vals, x)
    if case["op"] == "host":
        make = problems.laplace2d(*[int(k) for k in case["dims"].split("x")][::-1])
        make.data[:] = vals
        solver = SymLDLT()
        solver.setOrdering(OrderingType.AMD if case["ordering"] == "amd" else OrderingType.Metis)
        solver.analyzePattern(make)
        return dict(case=case, solver=solver, A=make, B=np.ascontiguousarray(b.cpu().numpy()).T)
    s = _System(patterns, case["ordering"])
    s.create()
    st = dict(case=case, system=s, vals=torch.from_numpy(vals).cuda(), b=b, x=torch.zeros_like(b),
              info=_lib.FactorInfo(), rinfo=_lib.RefineInfo(),
              per_system=(_lib.RefineInfo * len(patterns))(),
              ropts=_lib.RefineOpts(REFINE_ITERATIONS, REFINE_TOLERANCE), signs=None)
    if case["kind"] == "kkt":
        n1 = int(case["dims"]) ** 3
        st["signs"] = np.where(np.arange(n) < n1, -1, 1).astype(np.int32)
    st["opts"] = s.options(PRECISIONS[case["precision"]], st["signs"])
    torch.cuda.synchronize()
    if case["op"] == "solve":
        _factorize(st)
    elif case["op"] == "graph":
        args = (s.plan, _ptr(st["vals"]), _ptr(st["b"]), n, nrhs, _ptr(st["x"]), n, C.byref(st["opts"]))
        if case["refine"]:
            s._ok(s.lib.symla_graph_capture_refined(*args, C.byref(st["ropts"])))
        else:
            s._ok(s.lib.symla_graph_capture(*args))
    return st


def _factorize(st):
    s = st["system"]
    s._ok(s.lib.symla_factorize_device(s.plan, _ptr(st["vals"]), C.byref(st["opts"]), C.byref(st["info"])))


def _solve(st):
    s, n, nrhs = st["system"], st["system"].n, st["case"]["nrhs"]
    io = (_ptr(st["b"]), n, nrhs, _ptr(st["x"]), n)
    if not st["case"]["refine"]:
        s._ok(s.lib.symla_solve_device(s.plan, *io))
    elif len(s.sizes) > 1:
        s._ok(s.lib.symla_batch_solve_refined_device(s.plan, len(s.sizes), _lib.ptr(s.starts, _lib.i32p),
                                                     _ptr(st["vals"]), *io, C.byref(st["ropts"]), st["per_system"]))
    else:
        s._ok(s.lib.symla_solve_refined_device(s.plan, _ptr(st["vals"]), *io, C.byref(st["ropts"]),
                                               C.byref(st["rinfo"])))


def run(state):
    case = state["case"]
    if case["op"] == "host":
        solver = state["solver"]
        solver.refactorize(state["A"])
        x = solver.solve(state["B"])
        i = solver.inertia()
        return {"x": x.T, "inertia": [i.n_pos, i.n_neg, i.n_zero]}
    if case["op"] == "solve":
        _solve(state)
        return {"x": state["x"]}
    if case["op"] == "graph":
        s = state["system"]
        if case["refine"]:
            s._ok(s.lib.symla_graph_replay_refined(s.plan, C.byref(state["info"]), C.byref(state["rinfo"])))
        else:
            s._ok(s.lib.symla_graph_replay(s.plan, C.byref(state["info"])))
    else:
        _factorize(state)
        _solve(state)
    i = state["info"]
    return {"x": state["x"], "inertia": [i.n_pos, i.n_neg, i.n_zero]}


def exact(case, seed):
    """The solution that B was formed from without rounding."""
    x = _solution(_order(case)[1], case["nrhs"], seed)
    if case["op"] == "host":
        x = x.numpy()
    return {"x": x} if case["op"] == "solve" else {"x": x, "inertia": None}


@functools.lru_cache(maxsize=None)
def _factor_size(kind, dims, ordering):
    """(n, nnz(A), nnz(L), factor flops k m^2 - k^2 m + k^3 / 3 summed over the fronts) of the case's analysis."""
    s = _System(_patterns_cached((kind, dims)), ordering)
    info = _lib.SymbolicInfo()
    s._ok(s.lib.symla_symbolic_info(s.sym, C.byref(info)))
    first, ncols = np.empty(info.nsn, np.int32), np.empty(info.nsn, np.int32)
    perm, par = np.empty(info.n, np.int32), np.empty(info.n, np.int32)
    rp, rows = np.empty(info.nsn + 1, np.int64), np.empty(max(info.pattern_total, 1), np.int32)
    s._ok(s.lib.symla_symbolic_get(s.sym, _lib.ptr(perm, _lib.i32p), _lib.ptr(par, _lib.i32p),
                                   _lib.ptr(first, _lib.i32p), _lib.ptr(ncols, _lib.i32p),
                                   _lib.ptr(rp, _lib.i64p), _lib.ptr(rows, _lib.i32p)))
    m, k = np.diff(rp).astype(np.float64), ncols.astype(np.float64)
    nnz = sum(int(p[1][-1]) for p in _patterns_cached((kind, dims)))
    return info.n, nnz, int((m * k - k * (k - 1) / 2).sum()), float((k * m * m - k * k * m + k ** 3 / 3).sum())


def work(case):
    """Values and right-hand sides read, L written (a factorization) or read (a solve alone), solutions written."""
    n, nnz, nnzl, flops = _factor_size(case["kind"], case["dims"], case["ordering"])
    es = 8 if case["precision"] == "fp64" else 4
    solve = 4.0 * nnzl * case["nrhs"]
    return {"bytes": 8.0 * nnz * (case["op"] != "solve") + es * nnzl + 16.0 * n * case["nrhs"],
            "flops": solve + (flops if case["op"] != "solve" else 0.0)}
