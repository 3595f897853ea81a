"""The sync-free IC(0) factorization through the C-ABI.

Bars: factor and pivots bit-identical to the oracle at every row-length bucket
of the kernel and just past the longest it takes, real and complex; rows with
more updates than a wave holds at once; a replaced pivot; a factorization
forced to give up (spin limit 0 from the host) fails with HIP_ERROR, leaves no
factor behind, and the next one is right.
"""
import numpy as np
import pytest

from oracle import oracle as O
from sparsesolv_amd import capi

pytestmark = pytest.mark.gpu


def _banded(n, half, cplx, seed=0):
    """Symmetric, every row reading `half` rows on either side (a dense band: the most updates a row can have)."""
    rng = np.random.default_rng(seed)
    rp, ci = [0], []
    for i in range(n):
        ci.extend(range(max(0, i - half), min(n, i + half + 1)))
        rp.append(len(ci))
    rp, ci = np.asarray(rp, np.int32), np.asarray(ci, np.int32)
    row = np.repeat(np.arange(n), np.diff(rp))
    key = np.minimum(row, ci) * np.int64(n) + np.maximum(row, ci)
    _, inv = np.unique(key, return_inverse=True)
    v = rng.uniform(-1.0, 1.0, inv.max() + 1)[inv]
    if cplx:
        v = v + 1j * rng.uniform(-1.0, 1.0, inv.max() + 1)[inv]
    v[row == ci] = 4.0 * half
    return rp, ci, v


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("half", [0, 1, 19, 20, 31, 32, 47, 48])
def test_factor_bit_exact(torch_cuda, ctx, half, cplx):
    rp, ci, v = _banded(150, half, cplx)
    print(f"IC factor rows of {half + 1} entries cplx={cplx}", flush=True)
    m = capi.Matrix(ctx, rp, ci, v)
    try:
        got = m.ic_factor(1.1)
    finally:
        m.close()
    want = O.ic_decomp(rp, ci, v, 1.1)
    for a, b in zip(got[:4], want):
        assert np.array_equal(a, b)
    assert got[4] == np.count_nonzero(want[3] == 1.0 / np.finfo(float).eps)   # a lone zero diagonal: all replaced


def test_replaced_pivot(torch_cuda, ctx):
    rp, ci, v = _banded(40, 2, False)
    row = np.repeat(np.arange(40), np.diff(rp))
    v[(row == 20) | (ci == 20)] = 0.0   # row 20 stands alone with a zero pivot
    m = capi.Matrix(ctx, rp, ci, v)
    try:
        got = m.ic_factor(1.0)
    finally:
        m.close()
    want = O.ic_decomp(rp, ci, v, 1.0)
    for a, b in zip(got[:4], want):
        assert np.array_equal(a, b)
    assert got[4] == 1


def test_spin_limit_then_recovery(torch_cuda, ctx, monkeypatch):
    rp, ci, v = _banded(3000, 3, False)
    m = capi.Matrix(ctx, rp, ci, v)
    try:
        m.factorize(capi.ICCG, 1.1)
        print("factorization with spin limit 0", flush=True)
        monkeypatch.setenv("SSGPU_SPIN_LIMIT", "0")
        with pytest.raises(capi.SolverError) as e:
            m.factorize(capi.ICCG, 1.1)
        assert e.value.status == capi.HIP_ERROR
        monkeypatch.delenv("SSGPU_SPIN_LIMIT")
        d_r = torch_cuda.ones(m.n, dtype=torch_cuda.float64, device="cuda")
        with pytest.raises(capi.SolverError) as e:   # the failed factor is not used
            m.ic_apply_device(d_r.data_ptr(), d_r.data_ptr())
        assert e.value.status == capi.BAD_ARG
        got = m.ic_factor(1.1)
    finally:
        m.close()
    for a, b in zip(got[:4], O.ic_decomp(rp, ci, v, 1.1)):
        assert np.array_equal(a, b)
