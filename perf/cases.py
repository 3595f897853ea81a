"""The work a user of the solvers has them do, as cases that can be timed.

Each case is one pass through the public entry points of sparsesolv_amd on a
curl-curl edge-element system (voxel grid of n cells a side, N = 3 n (n-1)^2
unknowns): the kernel-level calls a program with its own Krylov loop makes,
the solves with a factor built once, the drop-in solve that refactors on every
call, several right-hand sides at once, many systems at once, and assembly.
Sizes are those of the tests (n = 6..16), of the served and batched workloads
(n = 8..60) and of the benchmark (n = 95).
"""
import math

import numpy as np
import torch

from sparsesolv_amd import assembly, capi, voxel

SOLVERS = {"iccg": capi.ICCG, "mrtr_ic": capi.MRTR_IC, "mrtr_sgs": capi.MRTR_SGS}
PRECISIONS = {"f64": capi.FACTOR_F64, "f32": capi.FACTOR_F32}
SHIFT = 1.2          # the benchmark's shift on the real systems
SHIFT_COMPLEX = 1.1  # and on the eddy-current systems
TOL = 1.0e-8
MAX_ITE = 2000
ABMC_BLOCK = 1

_context = None


def context():
    """One context for the whole program, as a program that solves one system after another keeps it."""
    global _context
    if _context is None:
        _context = capi.Context(0)
    return _context


# ----------------------------------------------------------------- the cases
def listed():
    return [
        # A program with its own Krylov loop asks for products at the benchmark's size: the streaming end.
        {"name": "spmv_n95", "kind": "spmv", "n": 95, "complex": False, "ordering": 0},
        # The same program's preconditioner on a small system: the latency of one call.
        {"name": "apply_n10", "kind": "apply", "n": 10, "complex": False, "ordering": 0},
        # Plain lower and upper triangular solves of an eddy-current matrix.
        {"name": "sweeps_complex_n32", "kind": "sweeps", "n": 32, "complex": True, "ordering": 0},
        # A nonlinear or time step: new values, a new factor, one application of it.
        {"name": "refactor_n40", "kind": "refactor", "n": 40, "complex": False, "ordering": 0},
        # The smallest whole solve: a cached factor, a few dozen iterations, launch and read-back latency.
        {"name": "iccg_n10", "kind": "factored", "n": 10, "complex": False, "ordering": 0, "solver": "iccg",
         "precision": "f64"},
        # The benchmark: the drop-in ICCG solve from host arrays, factorization included.
        {"name": "dropin_iccg_n95", "kind": "dropin", "n": 95, "complex": False, "ordering": 0, "solver": "iccg"},
        # The drop-in COCG solve of an eddy-current system.
        {"name": "dropin_cocg_n32", "kind": "dropin", "n": 32, "complex": True, "ordering": 0, "solver": "iccg"},
        # Eisenstat SGS-MRTR on the size of the served comparison.
        {"name": "sgs_n40", "kind": "factored", "n": 40, "complex": False, "ordering": 0, "solver": "mrtr_sgs",
         "precision": "f64"},
        # 32 excitations of one machine solved together.
        {"name": "block_mrtr_n40_rhs32", "kind": "block", "n": 40, "solver": "mrtr_ic", "rhs": 32},
        # Many independent small systems of uneven size in one batched session.
        {"name": "batch_iccg_16", "kind": "batch", "count": 16, "n": 8, "n_to": 24, "solver": "iccg"},
        # The multi-color order with its FP32 factor, for those who trade parity for speed.
        {"name": "abmc_f32_n60", "kind": "abmc", "n": 60, "precision": "f32"},
        # Element data to a resident matrix.
        {"name": "assemble_n40", "kind": "assemble", "n": 40, "complex": False},
    ]


def _size(rng, lo, hi):
    """A size between lo and hi, even over its logarithm where the range is wide."""
    if hi > 10 * lo:
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return rng.randint(lo, hi)


def draw(rng):
    kind = rng.choice(["spmv", "apply", "sweeps", "refactor", "factored", "factored", "dropin", "dropin", "block",
                       "batch", "abmc", "assemble"])
    cplx = rng.random() < 0.3
    ordering = 1 if rng.random() < 0.25 else 0
    if kind == "spmv":
        return {"kind": kind, "n": _size(rng, 10, 60 if cplx else 95), "complex": cplx, "ordering": ordering}
    if kind in ("apply", "sweeps"):
        return {"kind": kind, "n": _size(rng, 4, 40 if cplx else 60), "complex": cplx, "ordering": ordering}
    if kind == "refactor":
        return {"kind": kind, "n": _size(rng, 5, 48), "complex": cplx, "ordering": ordering}
    if kind == "factored":
        solver = "iccg" if cplx else rng.choice(sorted(SOLVERS))
        precision = "f64" if solver == "mrtr_sgs" else rng.choice(sorted(PRECISIONS))
        return {"kind": kind, "n": _size(rng, 5, 24 if cplx else 56), "complex": cplx, "ordering": ordering,
                "solver": solver, "precision": precision}
    if kind == "dropin":
        solver = "iccg" if cplx else rng.choice(sorted(SOLVERS))
        return {"kind": kind, "n": _size(rng, 6, 28 if cplx else 64), "complex": cplx, "ordering": ordering,
                "solver": solver}
    if kind == "block":
        return {"kind": kind, "n": _size(rng, 8, 36), "solver": rng.choice(sorted(SOLVERS)), "rhs": rng.randint(2, 32)}
    if kind == "batch":
        lo = rng.randint(6, 12)
        return {"kind": kind, "count": rng.randint(3, 16), "n": lo, "n_to": rng.randint(lo + 4, 28),
                "solver": rng.choice(sorted(SOLVERS))}
    if kind == "abmc":
        return {"kind": kind, "n": _size(rng, 16, 64), "precision": rng.choice(sorted(PRECISIONS))}
    return {"kind": kind, "n": _size(rng, 4, 44), "complex": cplx}


# --------------------------------------------------------------- the systems
def _system(case, seed):
    """The case's system: seeded materials and coil; at the benchmark's size its own fixed materials, as there."""
    n, ordering = case["n"], case.get("ordering", 0)
    if case.get("complex"):
        return voxel.eddy_current(n, seed=seed, ordering=ordering)
    materials = 0 if n >= 80 else seed
    return voxel.curlcurl(n, seed=materials, iron_fraction=0.2, ordering=ordering, coil_seed=seed + 1)


def _vector(seed, n, cplx):
    rng = np.random.default_rng(seed)
    v = rng.standard_normal(n)
    return v + 1j * rng.standard_normal(n) if cplx else v


def _shift(case):
    return SHIFT_COMPLEX if case.get("complex") else SHIFT


def _norm(b):
    return float(np.sqrt(np.sum(np.abs(b) ** 2)))


def _gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _triplets(case, seed):
    """Element data in the add order of the reference's assembly: (unknowns, rows, cols, values)."""
    n, cplx = case["n"], case["complex"]
    rng = np.random.default_rng(seed)
    mesh = voxel.tensor_mesh(*(np.linspace(0.0, 1.0, n + 1) for _ in range(3)))
    on_face = np.zeros(len(mesh.xyz), bool)
    for d in range(3):
        on_face |= (mesh.xyz[:, d] == 0.0) | (mesh.xyz[:, d] == 1.0)
    free = ~(on_face[mesh.edges[:, 0]] & on_face[mesh.edges[:, 1]])
    unknown = np.where(free, np.cumsum(free) - 1, -1)
    stiff, mass = voxel.element_matrices(1.0 / n)[:2]
    nu = rng.uniform(0.5, 1.5, len(mesh.elem_edges))
    ke = nu[:, None, None] * stiff[None]
    if cplx:
        ke = ke + 1j * rng.uniform(0.0, 1.0, len(nu))[:, None, None] * mass[None]
    rows, cols, vals = assembly.element_triplets(unknown[mesh.elem_edges], ke)
    return int(free.sum()), rows, cols, vals


# ------------------------------------------------------------------ a state
def prepare(case, seed):
    kind, ctx = case["kind"], context()
    if kind == "assemble":
        n, rows, cols, vals = _triplets(case, seed)
        return {"case": case, "n": n, "rows": _gpu(rows), "cols": _gpu(cols), "vals": _gpu(vals)}
    if kind == "batch":
        sizes = np.linspace(case["n"], case["n_to"], case["count"]).round().astype(int)
        code, mats, bs, xs, norms = SOLVERS[case["solver"]], [], [], [], []
        for k, n in enumerate(sizes):
            s = voxel.curlcurl(int(n), seed=1000 * seed + k, iron_fraction=0.2)
            m = capi.Matrix(ctx, s.row_ptr, s.col_idx, s.values)
            m.factorize(code, SHIFT)
            mats.append(m)
            bs.append(_gpu(s.rhs))
            xs.append(torch.zeros_like(bs[-1]))
            norms.append(_norm(s.rhs))
        return {"case": case, "mats": mats, "bs": bs, "xs": xs, "norms": norms, "solver": code}
    s = _system(case, seed)
    m = capi.Matrix(ctx, s.row_ptr, s.col_idx, s.values, abmc_block=ABMC_BLOCK if kind == "abmc" else None)
    state = {"case": case, "m": m}
    if kind in ("spmv", "apply", "sweeps", "refactor"):
        state["in"] = _gpu(_vector(seed, s.n, s.is_complex))
        state["out"] = torch.empty_like(state["in"])
        state["out2"] = torch.empty_like(state["in"])
        if kind == "apply":   # the call that builds a factor the kernel-level application may use
            m.factorize(capi.ICCG, _shift(case))
        if kind == "refactor":
            rng = np.random.default_rng(seed + 7)
            state["values"] = [s.values * f for f in rng.uniform(0.9, 1.1, 2)]
        return state
    if kind == "dropin":
        state.update(b=s.rhs, norm=_norm(s.rhs), solver=SOLVERS[case["solver"]],
                     opts=capi.default_options(is_save_log=1, accel_factor=_shift(case)))
        return state
    precision = PRECISIONS[case.get("precision", "f64")]
    code = SOLVERS[case.get("solver", "iccg")]
    state.update(solver=code, opts=capi.default_options(factor_precision=precision))
    m.factorize(code, _shift(case), precision)
    if kind == "block":
        rhs = np.stack([voxel.curlcurl(case["n"], seed=seed, iron_fraction=0.2, coil_seed=100 * seed + j).rhs
                        for j in range(case["rhs"])])
        state["norm"] = np.array([_norm(b) for b in rhs])
        state["b"] = _gpu(rhs)
    else:
        state["norm"] = _norm(s.rhs)
        state["b"] = _gpu(s.rhs)
    state["x"] = torch.zeros_like(state["b"])
    return state


def _solved(x, results):
    return {"x": x, "iterations": [r.iterations for r in results],
            "residuals": np.array([[r.final_residual, r.true_residual] for r in results])}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "assemble":
        m = capi.Matrix.from_triplets(context(), state["n"], state["rows"].data_ptr(), state["cols"].data_ptr(),
                                      state["vals"].data_ptr(), mode=capi.ASSEMBLE_BUILDER,
                                      ntrip=state["rows"].numel(), complex_=case["complex"])
        row_ptr, col_idx, values = m.csr()
        m.close()
        return {"row_ptr": row_ptr, "col_idx": col_idx, "values": values}
    if kind == "batch":
        res = capi.solve_batch(context(), state["mats"], [b.data_ptr() for b in state["bs"]],
                               [x.data_ptr() for x in state["xs"]], state["norms"], conv_cri=TOL, max_ite=MAX_ITE,
                               solver=state["solver"])
        return _solved(state["xs"], res)
    m = state["m"]
    if kind == "spmv":
        m.spmv_device(state["in"].data_ptr(), state["out"].data_ptr())
        return state["out"]
    if kind == "apply":
        m.ic_apply_device(state["in"].data_ptr(), state["out"].data_ptr())
        return state["out"]
    if kind == "sweeps":
        m.lower_sweep_device(state["in"].data_ptr(), state["out"].data_ptr())
        m.upper_sweep_device(state["in"].data_ptr(), state["out2"].data_ptr())
        return state["out"], state["out2"]
    if kind == "refactor":   # two sets of values in turn: every factor is of new ones
        outs = []
        for values, out in zip(state["values"], (state["out"], state["out2"])):
            m.update_values(values)
            m.factorize(capi.ICCG, _shift(case))
            m.ic_apply_device(state["in"].data_ptr(), out.data_ptr())
            outs.append(out)
        return outs
    if kind == "dropin":
        conv, x, log, res = m.solve(state["solver"], state["b"], conv_cri=TOL, max_ite=MAX_ITE, normB=state["norm"],
                                    opts=state["opts"])
        return dict(_solved(x, [res]), log=np.pad(log, (0, MAX_ITE + 2 - len(log))))
    if kind == "block":
        res = m.solve_block(context(), state["b"].data_ptr(), state["x"].data_ptr(), state["norm"],
                            solver=state["solver"], conv_cri=TOL, max_ite=MAX_ITE, opts=state["opts"])
        return _solved(state["x"], res)
    res = m.solve_factored(context(), state["solver"], state["b"].data_ptr(), state["x"].data_ptr(), conv_cri=TOL,
                           max_ite=MAX_ITE, normB=state["norm"], opts=state["opts"])
    return _solved(state["x"], [res])


# ------------------------------------------------------------ bytes and flops
def _unknowns(n):
    return 3 * n * (n - 1) ** 2


def _entries(n):
    """Entries of the matrix: an edge couples with the edges it shares a cell with."""
    same, cross = n * (3 * n - 5) ** 2, 2 * (2 * n - 2) * (2 * n - 2) * (3 * n - 5)
    return 3 * (same + cross)


def _one(n, kind, s_value, s_factor, columns=1):
    """(bytes, flops) of a product or of one triangular sweep (the sweeps of real and complex values alike)."""
    un, nz = _unknowns(n), _entries(n)
    ops = 2.0 if s_value == 8 else 8.0
    if kind == "spmv":
        return (s_value + 4.0) * nz + 4.0 * un + 2.0 * s_value * un * columns, ops * nz * columns
    low = (nz + un) // 2
    return ((s_factor + 4.0) * (low - un) + 4.0 * un + s_factor * un + 2.0 * s_value * un * columns,
            ops * low * columns)


def _krylov(n, iterations, solver, s_value=8, s_factor=8, columns=1):
    spmv, sweep = _one(n, "spmv", s_value, s_factor, columns), _one(n, "sweep", s_value, s_factor, columns)
    products = 0 if solver == "mrtr_sgs" else 1
    vectors = 10.0 * s_value * _unknowns(n) * columns   # x, r, p and the product, read and written once
    return (iterations * (products * spmv[0] + 2 * sweep[0] + vectors),
            iterations * (products * spmv[1] + 2 * sweep[1] + vectors / 4))


def work(case):
    """What one pass cannot do without; a solve is taken to need 2.4 n iterations (4 n on eddy-current systems),
    about what these systems take at this shift and tolerance."""
    kind, n, cplx = case["kind"], case["n"], case.get("complex", False)
    sv = 16 if cplx else 8
    its = (4.0 if cplx else 2.4) * n
    if kind == "spmv":
        b, f = _one(n, "spmv", sv, sv)
    elif kind in ("apply", "sweeps"):
        b, f = (2.0 * v for v in _one(n, "sweep", sv, sv))
    elif kind == "refactor":   # values in, a factor (read A's triangle, write L), two sweeps; twice
        sweep, low = _one(n, "sweep", sv, sv), (_entries(n) + _unknowns(n)) // 2
        b, f = 2.0 * (sv * _entries(n) + 2.0 * sv * low + 2 * sweep[0]), 2.0 * (30.0 * low + 2 * sweep[1])
    elif kind == "assemble":   # triplets in, the CSR matrix out
        trip = 144.0 * n ** 3
        b, f = (8.0 + sv) * trip + (4.0 + sv) * _entries(n) + 4.0 * _unknowns(n), sv / 8.0 * trip
    elif kind == "batch":
        sizes = np.linspace(case["n"], case["n_to"], case["count"]).round().astype(int)
        parts = [_krylov(int(k), 2.4 * int(k), case["solver"]) for k in sizes]
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    elif kind == "block":
        b, f = _krylov(n, its, case["solver"], columns=case["rhs"])
    else:
        sf = sv // 2 if case.get("precision") == "f32" else sv
        b, f = _krylov(n, its, case.get("solver", "iccg"), sv, sf)
    return {"bytes": float(b), "flops": float(f)}


# --------------------------------------------------------- values in 64 bits
def _product(s, x):
    return np.add.reduceat(s.values * x[s.col_idx], s.row_ptr[:-1])


def _triangular(rows, r, order):
    """x with x_i = (r_i - sum a_ij x_j) / d_i, rows[i] = (columns, values, diagonal), taken in the order given."""
    x = np.zeros_like(r)
    for i in order:
        cols, vals, d = rows[i]
        x[i] = (r[i] - (vals * x[cols]).sum()) / d
    return x


def _triangle(s, lower):
    rows = []
    for i in range(s.n):
        a, e = s.row_ptr[i], s.row_ptr[i + 1]
        cols, vals = s.col_idx[a:e], s.values[a:e]
        keep = cols < i if lower else cols > i
        rows.append((cols[keep], vals[keep], vals[cols == i][0]))
    return rows


def _factor(n, row_ptr, col_idx, values, shift):
    """Shifted root-free IC(0): per row its off-diagonal columns and values, its diagonal l_ii, and d_i = 1 / l_ii."""
    low, diag, d = [], [], []
    for i in range(n):
        a, e = row_ptr[i], row_ptr[i + 1]
        row, s = {}, None
        for c, v in zip(col_idx[a:e].tolist(), values[a:e].tolist()):
            if c > i:
                break
            acc = v * shift if c == i else v
            other = row if c == i else low[c]
            for k, l_ik in row.items():
                if k in other:
                    acc -= l_ik * other[k] * d[k]
            if c == i:
                s = acc
            else:
                row[c] = acc
        low.append(row)
        diag.append(s)
        d.append(1.0 / s)
    return low, diag, d


def _apply(n, row_ptr, col_idx, values, shift, r):
    """(L D L^T)^-1 r, L with its diagonal and D its inverse."""
    low, diag, d = _factor(n, row_ptr, col_idx, values, shift)
    y = [0.0] * n
    for i in range(n):
        acc = r[i]
        for k, v in low[i].items():
            acc = acc - v * y[k]
        y[i] = acc / diag[i]
    z, up = list(y), [0.0] * n
    for i in range(n - 1, -1, -1):
        z[i] = y[i] - d[i] * up[i]
        for k, v in low[i].items():
            up[k] = up[k] + v * z[i]
    return np.array(z)


def exact(case, seed):
    """What run returns, in 64 bits with plain numpy; None for the iterated solves, whose x no closed form gives (the
    systems are singular), and for factors that plain Python would take too long over."""
    kind = case["kind"]
    if kind == "assemble":
        n, rows, cols, vals = _triplets(case, seed)
        key = rows.astype(np.int64) * n + cols
        uniq, inv = np.unique(key, return_inverse=True)
        summed = np.zeros(len(uniq), vals.dtype)
        np.add.at(summed, inv, vals)
        row_ptr = np.searchsorted(uniq, np.arange(n + 1, dtype=np.int64) * n)
        return {"row_ptr": row_ptr.astype(np.int32), "col_idx": (uniq % n).astype(np.int32), "values": summed}
    if kind not in ("spmv", "apply", "sweeps", "refactor"):
        return None
    if kind in ("apply", "refactor") and case["n"] > 13:
        return None
    s = _system(case, seed)
    v = _vector(seed, s.n, s.is_complex)
    if kind == "spmv":
        return _product(s, v)
    if kind == "sweeps":
        return (_triangular(_triangle(s, True), v, range(s.n)),
                _triangular(_triangle(s, False), v, range(s.n - 1, -1, -1)))
    if kind == "apply":
        return _apply(s.n, s.row_ptr, s.col_idx, s.values, _shift(case), v)
    scale = np.random.default_rng(seed + 7).uniform(0.9, 1.1, 2)
    return [_apply(s.n, s.row_ptr, s.col_idx, s.values * f, _shift(case), v) for f in scale]
