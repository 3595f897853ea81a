"""Partitioned triangular sweeps (one workgroup per part of the rows, results
of a part handed over in LDS) through the C-ABI.

Bars: the plain lower and upper sweeps and the IC application are
bit-identical to the oracle and to the chunked sync-free shape for part sizes
from a few rows to the whole system, for grid cells, for every register bucket
of the row length, real and complex, FP64 and FP32 factors; divisors and
right-hand sides outside the range the precomputed reciprocal covers (and
zeros of both signs) give the quotients of plain division; a sweep forced to
give up (spin limit 0 from the host) fails with HIP_ERROR and the matrix then
solves as before.
"""
import time

import numpy as np
import pytest

from oracle import oracle as O
from sparsesolv_amd import capi, voxel

pytestmark = pytest.mark.gpu


def _lower(s):
    keep = np.concatenate([s[1][s[0][i]:s[0][i + 1]] <= i for i in range(len(s[0]) - 1)])
    rp = np.concatenate([[0], np.cumsum(np.add.reduceat(keep.astype(np.int64), s[0][:-1]))]).astype(np.int32)
    return rp, np.ascontiguousarray(s[1][keep]), np.ascontiguousarray(s[2][keep])


def _upper(s):
    keep = np.concatenate([s[1][s[0][i]:s[0][i + 1]] >= i for i in range(len(s[0]) - 1)])
    rp = np.concatenate([[0], np.cumsum(np.add.reduceat(keep.astype(np.int64), s[0][:-1]))]).astype(np.int32)
    return rp, np.ascontiguousarray(s[1][keep]), np.ascontiguousarray(s[2][keep])


def _run(torch, ctx, fn, r):
    d_r = torch.from_numpy(r).cuda()
    d_z = torch.zeros_like(d_r)
    torch.cuda.synchronize()
    fn(d_r.data_ptr(), d_z.data_ptr())
    ctx.synchronize()
    return d_z.cpu().numpy()


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


def _banded(n, length, cplx, seed=0):
    """A matrix whose rows read `length` rows on either side, near and far."""
    rng = np.random.default_rng(seed)
    step = np.unique(np.concatenate([[1, 2], 3 + np.sort(rng.choice(n // 3, max(0, length - 2), replace=False))]))
    step = step[:length]
    m = np.eye(n, dtype=bool)
    for d in step:
        i = np.arange(d, n)
        m[i, i - d] = m[i - d, i] = True
    rp, ci = [0], []
    for i in range(n):
        ci.extend(np.nonzero(m[i])[0].tolist())
        rp.append(len(ci))
    v = rng.uniform(-0.5, 0.5, len(ci))
    if cplx:
        v = v + 1j * rng.uniform(-0.5, 0.5, len(ci))
    rp, ci = np.asarray(rp, np.int32), np.asarray(ci, np.int32)
    v[np.concatenate([ci[rp[i]:rp[i + 1]] == i for i in range(n)])] = 4.0
    return rp, ci, v


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("length", [1, 8, 9, 13, 17, 20, 21, 25, 32])
def test_plain_sweeps_every_row_length(torch_cuda, ctx, monkeypatch, cplx, length):
    monkeypatch.setenv("SSGPU_SWEEP_MODE", "part")
    n = 700
    s = _banded(n, length, cplx)
    r = np.random.default_rng(1).standard_normal(n).astype(s[2].dtype)
    for rows in ("150", "700"):
        monkeypatch.setenv("SSGPU_PART_ROWS", rows)
        print(f"plain sweeps length={length} cplx={cplx} part rows={rows}", flush=True)
        m = capi.Matrix(ctx, *s)
        try:
            assert np.array_equal(_run(torch_cuda, ctx, m.lower_sweep_device, r), O.fr(_lower(s), r))
            assert np.array_equal(_run(torch_cuda, ctx, m.upper_sweep_device, r), O.bc(_upper(s), r))
        finally:
            m.close()


@pytest.mark.parametrize("n,cplx,env", [
    (4, False, {"SSGPU_PART_ROWS": "1"}), (6, False, {"SSGPU_PART_ROWS": "64"}), (7, True, {"SSGPU_PART_ROWS": "65"}),
    (13, False, {}), (20, False, {"SSGPU_PART_CELL": "3"}), (21, False, {}), (18, True, {"SSGPU_PART_CELL": "2"}),
    (24, False, {"SSGPU_PART_ROWS": "13000"})])
def test_ic_apply_equals_chunks_and_oracle(torch_cuda, ctx, monkeypatch, n, cplx, env):
    s = voxel.eddy_current(n, seed=2) if cplx else voxel.curlcurl(n, seed=2)
    r = np.random.default_rng(3).standard_normal(s.n).astype(s.values.dtype)
    out = []
    for mode in ("sf", "part"):
        monkeypatch.setenv("SSGPU_SWEEP_MODE", mode)
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        print(f"IC apply n={n} cplx={cplx} {mode} {env}", flush=True)
        m = capi.Matrix(ctx, s.row_ptr, s.col_idx, s.values)
        try:
            L = m.ic_factor(1.1)
            out.append(_run(torch_cuda, ctx, m.ic_apply_device, r))
            assert m.sweep_info()[0] == (3 if mode == "part" else 0)
        finally:
            m.close()
    ref = O.ic_apply(L[:3], O.transpose(L[0], L[1], L[2]), L[3], r)
    assert np.array_equal(_bits(out[0]), _bits(out[1]))
    assert np.array_equal(out[1], ref)


@pytest.mark.parametrize("solver", [capi.ICCG, capi.MRTR_IC, capi.MRTR_SGS], ids=["iccg", "mrtr_ic", "mrtr_sgs"])
@pytest.mark.parametrize("precision", [capi.FACTOR_F64, capi.FACTOR_F32], ids=["f64", "f32"])
def test_solves_equal_chunks(torch_cuda, ctx, monkeypatch, solver, precision):
    s = voxel.curlcurl(11, seed=5)
    out = []
    for mode in ("sf", "part"):
        monkeypatch.setenv("SSGPU_SWEEP_MODE", mode)
        monkeypatch.setenv("SSGPU_PART_ROWS", "500")
        print(f"solve solver={solver} precision={precision} {mode}", flush=True)
        m = capi.Matrix(ctx, s.row_ptr, s.col_idx, s.values)
        try:
            o = capi.default_options(accel_factor=1.2, is_save_log=1, factor_precision=precision)
            out.append(m.solve(solver, s.rhs, conv_cri=1e-8, max_ite=400, opts=o)[1:3])
        finally:
            m.close()
    assert np.array_equal(_bits(out[0][0]), _bits(out[1][0]))
    assert np.array_equal(out[0][1], out[1][1])


def test_quotients_outside_the_reciprocal_range(torch_cuda, ctx, monkeypatch):
    """Rows of a diagonal and a two-row coupling whose divisors and right-hand sides run over the whole
    exponent range, with zeros of both signs, infinities and NaN."""
    monkeypatch.setenv("SSGPU_SWEEP_MODE", "part")
    rng = np.random.default_rng(4)
    n = 4096
    d = rng.uniform(1.0, 2.0, n) * 2.0 ** rng.integers(-1021, 1022, n) * rng.choice([-1.0, 1.0], n)
    r = rng.uniform(1.0, 2.0, n) * 2.0 ** rng.integers(-1021, 1022, n) * rng.choice([-1.0, 1.0], n)
    r[:40:2], r[1:40:2] = 0.0, -0.0
    r[40:44] = [np.inf, -np.inf, np.nan, 5e-324]
    d[44:47] = [np.inf, -np.inf, 5e-324]
    rp, ci = np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32)
    m = capi.Matrix(ctx, rp, ci, d)
    try:
        with np.errstate(all="ignore"):
            ref = r / d
        for fn in (m.lower_sweep_device, m.upper_sweep_device):
            z = _run(torch_cuda, ctx, fn, r)
            nan = np.isnan(ref)
            assert np.array_equal(np.isnan(z), nan)
            assert np.array_equal(_bits(z[~nan]), _bits(ref[~nan]))
    finally:
        m.close()


def test_spin_limit_then_recovery(torch_cuda, ctx, monkeypatch):
    monkeypatch.setenv("SSGPU_SWEEP_MODE", "part")
    monkeypatch.setenv("SSGPU_PART_ROWS", "300")
    s = voxel.curlcurl(10, seed=6)
    o = capi.default_options(accel_factor=1.2, is_save_log=1)
    m = capi.Matrix(ctx, s.row_ptr, s.col_idx, s.values)
    try:
        ref = m.solve(capi.ICCG, s.rhs, conv_cri=1e-8, max_ite=300, opts=o)
        print("partitioned sweep with spin limit 0", flush=True)
        monkeypatch.setenv("SSGPU_SPIN_LIMIT", "0")
        with pytest.raises(capi.SolverError) as e:
            m.solve(capi.ICCG, s.rhs, conv_cri=1e-8, max_ite=300, opts=o)
        assert e.value.status == capi.HIP_ERROR
        monkeypatch.delenv("SSGPU_SPIN_LIMIT")
        again = m.solve(capi.ICCG, s.rhs, conv_cri=1e-8, max_ite=300, opts=o)
        assert np.array_equal(again[1], ref[1]) and np.array_equal(again[2], ref[2])
    finally:
        m.close()


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("solver,precision", [(capi.ICCG, capi.FACTOR_F64), (capi.MRTR_IC, capi.FACTOR_F32),
                                              (capi.MRTR_SGS, capi.FACTOR_F64), (capi.MRTR_SGS, capi.FACTOR_F32)])
def test_batch_of_every_sweep_kind_equals_chunks(torch_cuda, ctx, monkeypatch, cplx, solver, precision):
    """One batch whose systems sweep in parts of short rows, in parts of long rows and in chunks (rows of more
    than 32 entries), of one part and of many, against the same batch swept in chunks."""
    torch = torch_cuda
    systems = []
    for n, length in ((700, 4), (64, 20), (700, 21), (333, 32), (200, 40), (1, 1), (900, 20)):
        rp, ci, v = _banded(n, min(length, max(1, n // 4)), cplx, seed=n)
        v = np.where(v == 4.0, v, 0.05 * v)
        a = np.zeros((n, n), v.dtype)
        a[np.repeat(np.arange(n), np.diff(rp)), ci] = v
        a = a + a.T
        systems.append((rp, ci, np.ascontiguousarray(a[np.repeat(np.arange(n), np.diff(rp)), ci])))
    g = voxel.eddy_current(6, seed=3) if cplx else voxel.curlcurl(9, seed=3)
    systems.append((g.row_ptr, g.col_idx, g.values))
    rng = np.random.default_rng(8)
    rhs = [rng.standard_normal(len(s[0]) - 1).astype(s[2].dtype) for s in systems]
    opts = capi.default_options(factor_precision=precision)
    out = []
    for mode in ("sf", "part"):
        monkeypatch.setenv("SSGPU_SWEEP_MODE", mode)
        monkeypatch.setenv("SSGPU_PART_ROWS", "300")
        print(f"batch of sweep kinds solver={solver} precision={precision} cplx={cplx} {mode}", flush=True)
        mats = [capi.Matrix(ctx, *s) for s in systems]
        try:
            for m in mats:
                m.factorize(capi.ICCG if solver == capi.MRTR_IC else solver, 1.2, precision)
            d_b = [torch.from_numpy(b).cuda() for b in rhs]
            d_x = [torch.zeros_like(b) for b in d_b]
            torch.cuda.synchronize()
            res = capi.solve_batch(ctx, mats, [t.data_ptr() for t in d_b], [t.data_ptr() for t in d_x],
                                   [float(np.linalg.norm(b)) for b in rhs], solver=solver, conv_cri=1e-10,
                                   max_ite=60, opts=opts)
            out.append(([t.cpu().numpy() for t in d_x], [(r.converged, r.iterations, r.final_residual) for r in res]))
        finally:
            for m in mats:
                m.close()
    assert out[0][1] == out[1][1]
    for k, (a, b) in enumerate(zip(out[0][0], out[1][0])):
        assert np.array_equal(_bits(a), _bits(b)), k
    assert sum(i for _, i, _ in out[1][1]) > 40


def _wide(n, cplx):
    """Levels of hundreds of rows (steps of 64): one coupling, 300 rows apart."""
    rp, ci, v = [0], [], []
    for i in range(n):
        ci.extend(j for j in (i - 300, i, i + 300) if 0 <= j < n)
        rp.append(len(ci))
    ci = np.asarray(ci, np.int32)
    row = np.repeat(np.arange(n), np.diff(rp))
    v = np.where(ci == row, 4.0, 0.3 + 0.001 * ((row + ci) % 7))
    return np.asarray(rp, np.int32), ci, v * (1.0 + 0.25j) if cplx else v


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("solver,precision,kind,nrhs,rows", [
    (capi.ICCG, capi.FACTOR_F64, 4, 2, "150"), (capi.ICCG, capi.FACTOR_F32, 12, 3, "700"),
    (capi.MRTR_IC, capi.FACTOR_F64, 13, 1, "64"), (capi.MRTR_SGS, capi.FACTOR_F64, 20, 17, "150"),
    (capi.MRTR_SGS, capi.FACTOR_F32, 21, 32, "300"), (capi.ICCG, capi.FACTOR_F64, 32, 5, "1"),
    (capi.MRTR_IC, capi.FACTOR_F32, "wide", 4, "400"), (capi.MRTR_SGS, capi.FACTOR_F64, "grid", 6, "4000")])
def test_block_solves_equal_chunks(torch_cuda, ctx, monkeypatch, cplx, solver, precision, kind, nrhs, rows):
    """Two columns a workgroup and one (steps of more than 32 rows, one right-hand side, parts too large for
    two), every register bucket, against the chunked sweeps."""
    torch = torch_cuda
    if kind == "wide":
        s = _wide(1000, cplx)
    elif kind == "grid":
        g = voxel.eddy_current(12, seed=4) if cplx else voxel.curlcurl(12, seed=4)
        s = (g.row_ptr, g.col_idx, g.values)
    else:
        rp, ci, v = _banded(700, kind, cplx, seed=kind)
        row = np.repeat(np.arange(700), np.diff(rp))
        s = (rp, ci, np.where(ci == row, 8.0, 0.05 * np.cos(row + ci)).astype(v.dtype) * (1.0 + 0.2j if cplx else 1.0))
    n = len(s[0]) - 1
    b = np.random.default_rng(9).standard_normal((nrhs, n)).astype(s[2].dtype)
    opts = capi.default_options(factor_precision=precision)
    out = []
    for mode in ("sf", "part"):
        monkeypatch.setenv("SSGPU_SWEEP_MODE", mode)
        monkeypatch.setenv("SSGPU_PART_ROWS", rows)
        print(f"block solver={solver} precision={precision} {kind} nrhs={nrhs} cplx={cplx} {mode}", flush=True)
        m = capi.Matrix(ctx, *s)
        try:
            m.factorize(capi.ICCG if solver == capi.MRTR_IC else solver, 1.2, precision)
            d_b = torch.from_numpy(b).cuda()
            d_x = torch.zeros_like(d_b)
            torch.cuda.synchronize()
            res = m.solve_block(ctx, d_b.data_ptr(), d_x.data_ptr(), [float(np.linalg.norm(q)) for q in b],
                                solver=solver, conv_cri=1e-10, max_ite=25, opts=opts)
            out.append((d_x.cpu().numpy(), [(r.converged, r.iterations, r.final_residual) for r in res]))
        finally:
            m.close()
    assert out[0][1] == out[1][1]
    assert np.array_equal(_bits(out[0][0]), _bits(out[1][0]))


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("solver", [capi.ICCG, capi.MRTR_SGS], ids=["iccg", "mrtr_sgs"])
@pytest.mark.parametrize("kind,nrhs", [("chains", 3), ("chains", 12), ("chains", 30), ("long_rows", 2), ("long_rows", 7),
                                       ("long_rows", 16)])
def test_block_of_wide_levels_equals_chunks(torch_cuda, ctx, monkeypatch, cplx, solver, kind, nrhs):
    """Levels wide enough that small blocks sweep in parts and large ones in chunks."""
    torch = torch_cuda
    if kind == "chains":   # 400 chains of 25 rows
        n = 10000
        row = np.arange(n)
        pairs = [(row[1:][row[1:] % 25 != 0], -1)]
    else:                  # 30 levels of 400 rows, a row reading 10 of the level before
        n = 12000
        row = np.arange(n)
        pairs = [(row[400:], -400 - d if d else -400) for d in range(0, 10)]
        pairs = [(r[r + o >= (r // 400 - 1) * 400], o) for r, o in pairs]
    i = np.concatenate([r for r, _ in pairs])
    j = np.concatenate([r + o for r, o in pairs])
    i, j = np.concatenate([i, j, row]), np.concatenate([j, i, row])
    key = np.unique(i.astype(np.int64) * n + j)
    i, j = key // n, key % n
    rp = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=n))]).astype(np.int32)
    v = np.where(i == j, 25.0, -1.0 + 0.01 * ((i + j) % 5)) * (1.0 + 0.2j if cplx else 1.0)
    b = np.random.default_rng(nrhs).standard_normal((nrhs, n)).astype(v.dtype)
    out = []
    for mode in ("sf", None):
        if mode:
            monkeypatch.setenv("SSGPU_SWEEP_MODE", mode)
        else:
            monkeypatch.delenv("SSGPU_SWEEP_MODE")
        print(f"block of wide levels {kind} solver={solver} nrhs={nrhs} cplx={cplx} {mode}", flush=True)
        m = capi.Matrix(ctx, rp, j.astype(np.int32), v)
        try:
            m.factorize(solver, 1.2)
            d_b = torch.from_numpy(b).cuda()
            d_x = torch.zeros_like(d_b)
            torch.cuda.synchronize()
            res = m.solve_block(ctx, d_b.data_ptr(), d_x.data_ptr(), [float(np.linalg.norm(q)) for q in b],
                                solver=solver, conv_cri=1e-10, max_ite=25, opts=capi.default_options())
            out.append((d_x.cpu().numpy(), [(r.converged, r.iterations, r.final_residual) for r in res]))
        finally:
            m.close()
    assert out[0][1] == out[1][1]
    assert np.array_equal(_bits(out[0][0]), _bits(out[1][0]))


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("solver", [capi.ICCG, capi.MRTR_SGS], ids=["iccg", "mrtr_sgs"])
@pytest.mark.parametrize("copies", [5, 30])
def test_batch_of_wide_levels_equals_chunks(torch_cuda, ctx, monkeypatch, cplx, solver, copies):
    """Wide levels (50 intervals a system) beside narrow ones: few systems sweep in parts, many in chunks."""
    torch = torch_cuda
    n = 12000   # 30 levels of 400 rows, a row reading 5 of the level before
    row = np.arange(n)
    i = np.concatenate([row[400 + d:] for d in range(5)])
    j = np.concatenate([row[:n - 400 - d] for d in range(5)])
    i, j = i[j >= (i // 400 - 1) * 400], j[j >= (i // 400 - 1) * 400]
    i, j = np.concatenate([i, j, row]), np.concatenate([j, i, row])
    key = np.unique(i.astype(np.int64) * n + j)
    i, j = key // n, key % n
    rp = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=n))]).astype(np.int32)
    v = np.where(i == j, 15.0, -1.0 + 0.01 * ((i + j) % 5)) * (1.0 + 0.2j if cplx else 1.0)
    nr = _banded(700, 4, cplx)
    nr = (nr[0], nr[1], np.where(nr[2] == 4.0, 4.0, 0.1).astype(v.dtype))
    rng = np.random.default_rng(3)
    rhs = [rng.standard_normal(n).astype(v.dtype) for _ in range(copies)] + [rng.standard_normal(700).astype(v.dtype)]
    out = []
    for mode in ("sf", None):
        if mode:
            monkeypatch.setenv("SSGPU_SWEEP_MODE", mode)
        else:
            monkeypatch.delenv("SSGPU_SWEEP_MODE")
        print(f"batch of wide levels solver={solver} copies={copies} cplx={cplx} {mode}", flush=True)
        mats = [capi.Matrix(ctx, rp, j.astype(np.int32), v), capi.Matrix(ctx, *nr)]
        try:
            for m in mats:
                m.factorize(solver, 1.2)
            d_b = [torch.from_numpy(b).cuda() for b in rhs]
            d_x = [torch.zeros_like(b) for b in d_b]
            torch.cuda.synchronize()
            res = capi.solve_batch(ctx, [mats[0]] * copies + [mats[1]], [t.data_ptr() for t in d_b],
                                   [t.data_ptr() for t in d_x], [float(np.linalg.norm(b)) for b in rhs],
                                   solver=solver, conv_cri=1e-10, max_ite=30, opts=capi.default_options())
            out.append(([t.cpu().numpy() for t in d_x], [(r.converged, r.iterations, r.final_residual) for r in res]))
        finally:
            for m in mats:
                m.close()
    assert out[0][1] == out[1][1]
    for k, (a, b) in enumerate(zip(out[0][0], out[1][0])):
        assert np.array_equal(_bits(a), _bits(b)), k


@pytest.mark.parametrize("mode,kind", [("sf", 0), ("level", 1), ("tile", 2), ("part", 3)])
@pytest.mark.parametrize("n", [5, 8, 13])
def test_shape_asked_for_after_creation(torch_cuda, ctx, monkeypatch, n, mode, kind):
    """A shape asked for at the first factorization runs, whatever the creation built, with the same bits."""
    s = voxel.curlcurl(n, seed=6)
    o = capi.default_options(accel_factor=1.2, is_save_log=1)
    out = []
    for env in (None, mode):
        m = capi.Matrix(ctx, s.row_ptr, s.col_idx, s.values)
        try:
            if env:
                monkeypatch.setenv("SSGPU_SWEEP_MODE", env)
            print(f"n={n} shape after creation: {env}", flush=True)
            out.append(m.solve(capi.ICCG, s.rhs, conv_cri=1e-8, max_ite=300, opts=o)[1:3])
            out.append(m.solve(capi.ICCG, s.rhs, conv_cri=1e-8, max_ite=300, opts=o)[1:3])
            assert m.sweep_info()[0] == (kind if env else 3)
            out.append(m.solve(capi.MRTR_SGS, s.rhs, conv_cri=1e-8, max_ite=40, opts=o)[1:3])
        finally:
            m.close()
    for a, b in zip(out[:3], out[3:]):
        assert np.array_equal(_bits(a[0]), _bits(b[0])) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("precision", [capi.FACTOR_F64, capi.FACTOR_F32], ids=["f64", "f32"])
def test_tuner_that_takes_chunks(torch_cuda, ctx, monkeypatch, cplx, precision):
    """Levels wide enough for the tuner to time parts against chunks, forced to chunks after both were built: the
    IC sweeps leave the parts, SGS sweeps mix chunks forward and parts backward, and block and batched solves follow."""
    torch = torch_cuda
    n = 14400   # 24 levels of 600 rows, a row reading 5 of the level before
    row = np.arange(n)
    i = np.concatenate([row[600 + d:] for d in range(5)])
    j = np.concatenate([row[:n - 600 - d] for d in range(5)])
    i, j = i[j >= (i // 600 - 1) * 600], j[j >= (i // 600 - 1) * 600]
    i, j = np.concatenate([i, j, row]), np.concatenate([j, i, row])
    key = np.unique(i.astype(np.int64) * n + j)
    i, j = key // n, key % n
    rp = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=n))]).astype(np.int32)
    v = np.where(i == j, 15.0, -1.0 + 0.01 * ((i + j) % 5)) * (1.0 + 0.2j if cplx else 1.0)
    b = np.random.default_rng(4).standard_normal((3, n)).astype(v.dtype)
    norms = [float(np.linalg.norm(q)) for q in b]
    opts = capi.default_options(factor_precision=precision)
    out = []
    for chunks in (False, True):
        monkeypatch.delenv("SSGPU_SWEEP_MODE", raising=False)
        if not chunks:
            monkeypatch.setenv("SSGPU_SWEEP_MODE", "part")
        m = capi.Matrix(ctx, rp, j.astype(np.int32), v)
        got = []
        try:
            if chunks:
                monkeypatch.setenv("SSGPU_SWEEP_MODE", "sf")
            for solver in (capi.ICCG, capi.MRTR_SGS, capi.MRTR_IC):
                print(f"tuner takes chunks={chunks} solver={solver} precision={precision} cplx={cplx}", flush=True)
                m.factorize(solver if solver == capi.MRTR_SGS else capi.ICCG, 1.2, precision)
                assert m.sweep_info()[0] == (0 if chunks else 3)
                d_b = torch.from_numpy(b).cuda()
                d_x = torch.zeros_like(d_b)
                torch.cuda.synchronize()
                res = [m.solve_factored(ctx, solver, d_b[0].data_ptr(), d_x[0].data_ptr(), conv_cri=1e-10, max_ite=20,
                                        normB=norms[0], opts=opts)]
                got.append((d_x.cpu().numpy(), [(r.converged, r.iterations, r.final_residual) for r in res]))
                res = m.solve_block(ctx, d_b.data_ptr(), d_x.data_ptr(), norms, solver=solver, conv_cri=1e-10,
                                    max_ite=20, opts=opts)
                got.append((d_x.cpu().numpy(), [(r.converged, r.iterations, r.final_residual) for r in res]))
                res = capi.solve_batch(ctx, [m] * 3, [q.data_ptr() for q in d_b], [q.data_ptr() for q in d_x], norms,
                                       solver=solver, conv_cri=1e-10, max_ite=20, opts=opts)
                got.append((d_x.cpu().numpy(), [(r.converged, r.iterations, r.final_residual) for r in res]))
        finally:
            m.close()
        out.append(got)
    for a, c in zip(*out):
        assert a[1] == c[1]
        assert np.array_equal(_bits(a[0]), _bits(c[0]))


def test_failed_sweep_ends_without_its_later_parts(torch_cuda, ctx, monkeypatch):
    """A chain in 2000 parts: with a limit shorter than the wait of the last parts on the GPU at once, the sweep fails,
    and the parts that have not started by then do not wait in their turn (8 or more rounds of that limit, which
    together take most of the time of the whole sweep)."""
    n = 300000
    rp = np.concatenate([[0], np.cumsum(np.where((np.arange(n) == 0) | (np.arange(n) == n - 1), 2, 3))]).astype(np.int32)
    row = np.repeat(np.arange(n), np.diff(rp))
    first = rp[:-1][row]
    ci = (np.arange(len(row)) - first + np.maximum(row - 1, 0)).astype(np.int32)
    monkeypatch.setenv("SSGPU_PART_ROWS", "150")
    m = capi.Matrix(ctx, rp, ci, np.where(ci == row, 2.01, -1.0))
    r = torch_cuda.ones(n, dtype=torch_cuda.float64, device="cuda")
    z = torch_cuda.zeros_like(r)

    def sweep():
        torch_cuda.cuda.synchronize()
        t = time.perf_counter()
        try:
            m.lower_sweep_device(r.data_ptr(), z.data_ptr())
            return time.perf_counter() - t, capi.OK
        except capi.SolverError as e:
            return time.perf_counter() - t, e.status

    try:
        print("chain in 2000 parts, whole sweep", flush=True)
        whole = [sweep() for _ in range(3)]
        ref = z.cpu().numpy()
        print("the same with a spin limit of 6000 passes", flush=True)
        monkeypatch.setenv("SSGPU_SPIN_LIMIT", "6000")
        failed = sweep()
        monkeypatch.delenv("SSGPU_SPIN_LIMIT")
        again = sweep()
    finally:
        m.close()
    print(f"whole {whole}, failed {failed}", flush=True)
    assert all(s == capi.OK for _, s in whole + [again])
    assert np.array_equal(z.cpu().numpy(), ref)
    assert failed[1] == capi.HIP_ERROR
    assert failed[0] < 0.4 * min(t for t, _ in whole)


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("solver", [capi.ICCG, capi.MRTR_SGS], ids=["iccg", "mrtr_sgs"])
@pytest.mark.parametrize("order", ["ic_first", "sgs_first"])
def test_parts_in_one_direction_only(torch_cuda, ctx, monkeypatch, cplx, solver, order):
    """Rows short enough for parts below the diagonal, and too long above it: 100 groups of 50 rows that read their
    group's first row, which reads the group's before."""
    torch = torch_cuda
    n = 5000
    row = np.arange(n)
    head = row // 50 * 50
    i = np.concatenate([row[row != head], head[50::50]])
    j = np.concatenate([head[row != head], head[50::50] - 50])
    i, j = np.concatenate([i, j, row]), np.concatenate([j, i, row])
    key = np.unique(i.astype(np.int64) * n + j)
    i, j = key // n, key % n
    rp = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=n))]).astype(np.int32)
    v = np.where(i == j, 60.0, -1.0 + 0.01 * ((i + j) % 5)) * (1.0 + 0.2j if cplx else 1.0)
    b = np.random.default_rng(5).standard_normal((2, n)).astype(v.dtype)
    norms = [float(np.linalg.norm(q)) for q in b]
    out = []
    for mode in ("sf", None):
        if mode:
            monkeypatch.setenv("SSGPU_SWEEP_MODE", mode)
        else:
            monkeypatch.delenv("SSGPU_SWEEP_MODE")
        print(f"parts below the diagonal only, solver={solver} {order} cplx={cplx} {mode}", flush=True)
        m = capi.Matrix(ctx, rp, j.astype(np.int32), v)
        try:
            m.factorize(capi.MRTR_SGS if order == "sgs_first" else capi.ICCG, 1.2)
            m.factorize(solver, 1.2)
            d_b = torch.from_numpy(b).cuda()
            d_x = torch.zeros_like(d_b)
            torch.cuda.synchronize()
            res = [m.solve_factored(ctx, solver, d_b[0].data_ptr(), d_x[0].data_ptr(), conv_cri=1e-10, max_ite=30,
                                    normB=norms[0], opts=capi.default_options())]
            solo = d_x[0].cpu().numpy()
            res += capi.solve_batch(ctx, [m] * 2, [q.data_ptr() for q in d_b], [q.data_ptr() for q in d_x], norms,
                                    solver=solver, conv_cri=1e-10, max_ite=30, opts=capi.default_options())
            out.append((solo, d_x.cpu().numpy(), [(r.converged, r.iterations, r.final_residual) for r in res]))
        finally:
            m.close()
    assert out[0][2] == out[1][2]
    assert np.array_equal(_bits(out[0][0]), _bits(out[1][0]))
    assert np.array_equal(_bits(out[0][1]), _bits(out[1][1]))


@pytest.mark.parametrize("n,mode", [(20, None), (20, "sf")])
def test_calls_in_place(torch_cuda, ctx, monkeypatch, n, mode):
    """An application and plain sweeps whose result takes the place of the right-hand side, after a whole solve."""
    if mode:
        monkeypatch.setenv("SSGPU_SWEEP_MODE", mode)
    s = voxel.curlcurl(n, seed=2, ordering=1)
    r = np.random.default_rng(6).standard_normal(s.n)
    m = capi.Matrix(ctx, s.row_ptr, s.col_idx, s.values)
    try:
        print(f"in place n={n} {mode}", flush=True)
        m.solve(capi.ICCG, s.rhs, conv_cri=1e-8, max_ite=50, opts=capi.default_options(accel_factor=1.2))
        for fn in (m.ic_apply_device, m.lower_sweep_device, m.upper_sweep_device):
            want = _run(torch_cuda, ctx, fn, r)
            d = torch_cuda.from_numpy(r).cuda()
            torch_cuda.cuda.synchronize()
            fn(d.data_ptr(), d.data_ptr())
            ctx.synchronize()
            assert np.array_equal(_bits(d.cpu().numpy()), _bits(want))
    finally:
        m.close()
