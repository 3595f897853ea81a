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


def _layers(width, length, cplx):
    """Four wide levels; a row of level l reads rows of the levels below it that share columns among themselves."""
    rng = np.random.default_rng(length)
    n = 4 * width
    reads = [np.zeros(0, np.int64)] * width
    for lev in range(1, 4):
        for k in range(width):
            base = k // length * length   # neighbours read the same rows, so that updates exist
            below = (base + rng.permutation(2 * length)[:length]) % width + width * rng.integers(0, lev, length)
            below[0] = (lev - 1) * width + k
            reads.append(np.unique(below))
    row = np.concatenate([np.full(len(c), i) for i, c in enumerate(reads)] + [np.arange(n)])
    col = np.concatenate(reads + [np.arange(n)])
    val = rng.uniform(-1.0, 1.0, len(row)) + (1j * rng.uniform(-1.0, 1.0, len(row)) if cplx else 0.0)
    val[row == col] = 3.0 * length
    off = row != col
    i, j, v = np.concatenate([row, col[off]]), np.concatenate([col, row[off]]), np.concatenate([val, val[off]])
    order = np.lexsort((j, i))
    rp = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=n))]).astype(np.int32)
    return rp, j[order].astype(np.int32), v[order]


@pytest.mark.parametrize("cplx,width", [(False, 2999), (False, 3000), (False, 3203), (True, 1499), (True, 1501)])
@pytest.mark.parametrize("length", [3, 19, 20, 31, 47])
def test_wide_levels_bit_exact(torch_cuda, ctx, cplx, width, length):
    """Both sides of the width from which a level is a launch of its own, every bucket of the row length."""
    rp, ci, v = _layers(width, length, cplx)
    print(f"IC factor of 4 levels of {width} rows, {length} entries below, cplx={cplx}", flush=True)
    m = capi.Matrix(ctx, rp, ci, v)
    try:
        assert m.info()["fwd_levels"] == 4
        got = m.ic_factor(1.1)
    finally:
        m.close()
    want = O.ic_decomp(rp, ci, v, 1.1)
    for a, b in zip(got[:4], want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
def test_any_nan_in_the_matrix_is_factored(torch_cuda, ctx, cplx):
    """Entries of every kind of NaN, the bits that the kernels wait on among them: the factor has NaN where the
    oracle's has it, and the other values its bits; denormal and signed-zero entries stay as they are."""
    rp, ci, v = _banded(60, 1, cplx)
    row = np.repeat(np.arange(60), np.diff(rp))
    bits = [0xFFF40000DEADBEEF, 0x7FF0000000000001, 0x7FF8000000000000, 0xFFF8000000000000]
    part = v.view(np.float64).reshape(len(v), -1)[:, -1]
    for k, b in enumerate(bits):
        i = 10 * (k + 1)
        part[(row == i) & (ci == i - 1)] = part[(row == i - 1) & (ci == i)] = np.uint64(b).view(np.float64)
    v[(row == 55) & (ci == 54)] = v[(row == 54) & (ci == 55)] = 5e-324
    v[(row == 57) & (ci == 56)] = v[(row == 56) & (ci == 57)] = -0.0
    print(f"IC factor of a matrix with NaN entries cplx={cplx}", flush=True)
    m = capi.Matrix(ctx, rp, ci, v)
    try:
        got = m.ic_factor(1.1)
    finally:
        m.close()
    want = O.ic_decomp(rp, ci, v, 1.1)
    for a, b in zip(got[2:4], want[2:4]):
        a, b = a.view(np.float64), b.view(np.float64)
        nan = np.isnan(b)
        assert nan.any() and not nan.all()
        assert np.array_equal(np.isnan(a), nan)
        assert np.array_equal(a[~nan].view(np.uint64), b[~nan].view(np.uint64))
