"""Device-memory controls: ssgpu_context_trim, ssgpu_batch_trim, ssgpu_memory.

A trimmed context holds exactly its matrices' bytes again and its next solve
is bit-identical to the one before the trim (the pool is regrown); a batch
session that has drained gives its slot vectors back; the library's counters
agree with the contexts' own.
"""
import numpy as np
import pytest

from sparsesolv_amd import capi, serve, voxel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", [capi.ICCG, capi.MRTR_IC, capi.MRTR_SGS], ids=["iccg", "mrtr_ic", "mrtr_sgs"])
def test_trim_frees_the_pool_and_solves_the_same(torch_cuda, solver):
    torch = torch_cuda
    s = voxel.curlcurl(12, seed=3)
    print(f"trim solver={solver} N={s.n}", flush=True)
    ctx = capi.Context(0)
    m = capi.Matrix(ctx, s.row_ptr, s.col_idx, s.values)
    try:
        m.factorize(solver, 1.1)
        held = ctx.resident_bytes()
        d_b = torch.from_numpy(s.rhs.copy()).cuda()
        o = capi.default_options(accel_factor=1.1, is_save_best=1)

        def solve():
            d_x = torch.zeros_like(d_b)
            torch.cuda.synchronize()
            r = m.solve_factored(ctx, solver, d_b.data_ptr(), d_x.data_ptr(), conv_cri=1e-8, max_ite=2000,
                                 normB=float(np.linalg.norm(s.rhs)), opts=o)
            return d_x.cpu().numpy(), r

        x1, r1 = solve()
        grown = ctx.resident_bytes()
        assert grown > held   # the work pool
        assert grown - held <= serve._pool_bytes(s.n, False)
        now, peak = capi.memory()
        assert peak >= now >= grown
        ctx.trim()
        # left: the matrices, and the context's scalar block if the first solve made it
        base = ctx.resident_bytes()
        assert held <= base <= held + 4096
        assert capi.memory()[0] == now - (grown - base)
        x2, r2 = solve()
        assert r2.iterations == r1.iterations
        assert np.array_equal(x1, x2)
        assert ctx.resident_bytes() == grown
        ctx.trim()
        assert ctx.resident_bytes() == base
    finally:
        m.close()
        ctx.close()


def test_batch_trim_returns_slot_vectors(torch_cuda, ctx):
    systems = [voxel.curlcurl(9, seed=11), voxel.curlcurl(13, seed=12)]
    print(f"batch trim N={[s.n for s in systems]}", flush=True)
    mats = [capi.Matrix(ctx, s.row_ptr, s.col_idx, s.values) for s in systems]
    c2 = capi.Context(0)
    b = capi.Batch(c2, False, capi.FACTOR_F64)
    try:
        for m in mats:
            m.factorize(capi.ICCG, 1.1)
        o = capi.default_options(accel_factor=1.1)
        base = c2.resident_bytes()
        xs = [np.zeros(s.n) for s in systems]
        for t, (s, m, x) in enumerate(zip(systems, mats, xs)):
            b.add_host(m, np.ascontiguousarray(s.rhs), x, t, normB=float(np.linalg.norm(s.rhs)), conv_cri=1e-8,
                       max_ite=2000, opts=o)
        vec_bytes = sum(serve._batch_vector_bytes(s.n, False) for s in systems)
        assert c2.resident_bytes() - base <= vec_bytes + (1 << 20)   # slots plus the session's tables
        got = {}
        for _ in range(1000):
            running, _ = b.step(8)
            got.update(dict(b.poll()))
            if running == 0:
                break
        assert sorted(got) == [0, 1] and all(r.converged for r in got.values())
        before = c2.resident_bytes()
        b.trim()
        c2.trim()
        after = c2.resident_bytes()
        slots = sum(8 * 8 * s.n for s in systems)
        assert before - after >= slots
        # the session still serves: one more system after the trim, same answer as before
        x_again = np.zeros(systems[0].n)
        b.add_host(mats[0], np.ascontiguousarray(systems[0].rhs), x_again, 7,
                   normB=float(np.linalg.norm(systems[0].rhs)), conv_cri=1e-8, max_ite=2000, opts=o)
        res = {}
        for _ in range(1000):
            running, _ = b.step(8)
            res.update(dict(b.poll()))
            if running == 0:
                break
        assert res[7].iterations == got[0].iterations
        assert np.array_equal(x_again, xs[0])
    finally:
        b.close()
        c2.close()
        for m in mats:
            m.close()


def _symmetric(n, offsets, period=0):
    """Couplings a fixed number of rows apart, none across multiples of the period."""
    row = np.arange(n)
    i = np.concatenate([row[d:] for d in offsets])
    j = np.concatenate([row[:n - d] for d in offsets])
    if period:
        i, j = i[i % period != 0], j[i % period != 0]
    i, j = np.concatenate([i, j, row]), np.concatenate([j, i, row])
    key = np.unique(i.astype(np.int64) * n + j)
    i, j = key // n, key % n
    rp = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=n))]).astype(np.int32)
    return rp, j.astype(np.int32), np.where(i == j, 2.0 * len(offsets) + 0.5, -1.0)


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("kind", ["diagonal", "chain", "chains", "strip", "grid", "edge_natural", "edge_blocked",
                                  "edge_colors", "edge_color_blocks"])
def test_building_stays_within_the_serving_bound(torch_cuda, kind, cplx):
    """The peak of creation and factorization, for every solver and factor precision, stays within what the serving
    engine reserves for it."""
    block = {"edge_colors": 1, "edge_color_blocks": 16}.get(kind)
    if kind.startswith("edge"):
        s = voxel.curlcurl(18, seed=2, ordering=1 if kind == "edge_blocked" else 0)
        rp, ci, v = s.row_ptr, s.col_idx, s.values
    else:
        rp, ci, v = {"diagonal": lambda: _symmetric(30000, [0]), "chain": lambda: _symmetric(30000, [1]),
                     "chains": lambda: _symmetric(60000, [1], 40), "strip": lambda: _symmetric(40000, [1, 8]),
                     "grid": lambda: _symmetric(90000, [1, 300])}[kind]()
    if cplx:
        v = v * (1.0 + 0.2j)
    worst = 0.0
    for solver in (capi.ICCG, capi.MRTR_SGS):
        for precision in (capi.FACTOR_F64, capi.FACTOR_F32):
            print(f"serving bound {kind} cplx={cplx} solver={solver} precision={precision}", flush=True)
            c = capi.Context(0)
            base = capi.memory(reset_peak=True)[0]
            m = capi.Matrix(c, rp, ci, v, abmc_block=block)
            try:
                m.factorize(solver, 1.2, precision)
                peak = capi.memory()[1] - base
            finally:
                m.close()
                c.close()
            worst = max(worst, peak / serve._system_bytes(len(ci), len(rp) - 1, cplx, precision))
    print(f"  at most {worst:.2f} of the bound", flush=True)
    assert worst <= 1.0
