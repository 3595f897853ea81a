"""The dot products and norms of block solves (a row's columns side by side, one lane per row and column).

Bar: every column of a block solve has the bits of its solo solve, whose sums
run over one column, at row counts around the edges of waves, workgroups and
the reduction grid, for every padded column count, real and complex.
"""
import numpy as np
import pytest

from sparsesolv_amd import capi

pytestmark = pytest.mark.gpu


def _coupled(n, cplx):
    """Diagonally dominant, one coupling 7 rows apart."""
    row = np.concatenate([np.arange(n), np.arange(7, n), np.arange(n - 7) if n > 7 else np.arange(0)])
    col = np.concatenate([np.arange(n), np.arange(n - 7) if n > 7 else np.arange(0), np.arange(7, n)])
    order = np.lexsort((col, row))
    row, col = row[order], col[order]
    v = np.where(row == col, 4.0 + (row % 5) * 0.25, 0.3 + 0.01 * ((row + col) % 11))
    rp = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))]).astype(np.int32)
    return rp, col.astype(np.int32), v * (1.0 + 0.25j) if cplx else v


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("n,nrhs", [(1, 1), (63, 2), (64, 3), (65, 32), (255, 8), (257, 16), (1000, 31),
                                    (262144 + 65, 5)])
@pytest.mark.parametrize("solver", [capi.ICCG, capi.MRTR_IC], ids=["iccg", "mrtr_ic"])
def test_columns_equal_solo(torch_cuda, ctx, n, nrhs, cplx, solver):
    torch = torch_cuda
    s = _coupled(n, cplx)
    rng = np.random.default_rng(n + nrhs)
    b = rng.standard_normal((nrhs, n)).astype(s[2].dtype)
    if cplx:
        b = b + 1j * rng.standard_normal((nrhs, n))
    norms = [float(np.linalg.norm(q)) for q in b]
    opts = capi.default_options()
    print(f"block reductions n={n} nrhs={nrhs} cplx={cplx} solver={solver}", flush=True)
    m = capi.Matrix(ctx, *s)
    try:
        m.factorize(capi.ICCG, 1.1, capi.FACTOR_F64)
        d_b = torch.from_numpy(b).cuda()
        d_x = torch.zeros_like(d_b)
        torch.cuda.synchronize()
        res = m.solve_block(ctx, d_b.data_ptr(), d_x.data_ptr(), norms, solver=solver, conv_cri=1e-14, max_ite=4,
                            opts=opts)
        for j in sorted({0, nrhs // 2, nrhs - 1}):
            x = torch.zeros_like(d_b[j])
            torch.cuda.synchronize()
            r = m.solve_factored(ctx, solver, d_b[j].data_ptr(), x.data_ptr(), conv_cri=1e-14, max_ite=4,
                                 normB=norms[j], opts=opts)
            ctx.synchronize()
            assert (r.iterations, r.final_residual) == (res[j].iterations, res[j].final_residual), j
            assert np.array_equal(x.cpu().numpy().view(np.uint64), d_x[j].cpu().numpy().view(np.uint64)), j
    finally:
        m.close()
