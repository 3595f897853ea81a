"""Layout of the partitioned sweeps (ssgpu_parts.h) on the CPU.

tests/cpp/part_layout_main.cpp walks a layout as the kernel does and checks
each index; the solution it forms must be bit-identical to a plain triangular
solve in the reference's order (the oracle), for intervals and grid cells,
both directions, on grids, chains, scattered and edge-case patterns.  The
quotient from a known reciprocal is compared with division.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle import oracle as O
from sparsesolv_amd import voxel

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("part") / "libpart.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", "-shared", "-fPIC", "-pthread",
                    f"-I{ROOT}/sparsesolv_amd/csrc", os.path.join(ROOT, "tests", "cpp", "part_layout_main.cpp"),
                    "-o", out], check=True)
    return ctypes.CDLL(out)


def _dense_pattern(n, mask):
    rp, ci = [0], []
    for i in range(n):
        ci.extend(np.nonzero(mask[i])[0].tolist())
        rp.append(len(ci))
    return np.asarray(rp, np.int32), np.asarray(ci, np.int32)


def _matrix(kind):
    rng = np.random.default_rng(5)
    if kind == "grid":
        s = voxel.curlcurl(20, seed=1)
        return s.n, s.row_ptr, s.col_idx, s.values
    if kind == "direction_blocked":
        s = voxel.curlcurl(9, seed=1, ordering=1)
        return s.n, s.row_ptr, s.col_idx, s.values
    n = {"one": 1, "diagonal": 300, "chain": 500, "scattered": 700, "wide": 900}[kind]
    m = np.eye(n, dtype=bool)
    if kind == "chain":
        m |= np.eye(n, k=1, dtype=bool) | np.eye(n, k=-1, dtype=bool)
    if kind == "scattered":
        m |= rng.random((n, n)) < 0.01
        m |= m.T
    if kind == "wide":   # rows that read many rows of a first, independent block
        for i in range(300, n):
            m[i, rng.choice(300, 20, replace=False)] = True
        m |= m.T
    rp, ci = _dense_pattern(n, m)
    v = rng.uniform(0.5, 1.5, len(ci))
    return n, rp, ci, v


def _reference(n, rp, ci, v, r, forward):
    x = np.zeros(n)
    for i in (range(n) if forward else range(n - 1, -1, -1)):
        acc, d = r[i], 1.0
        for k in range(rp[i], rp[i + 1]):
            j = ci[k]
            if j == i:
                d = v[k]
            elif (j < i) == forward:
                acc = acc - v[k] * x[j]
        x[i] = acc / d
    return x


@pytest.mark.parametrize("kind,rows,cell", [
    ("one", 5, 0), ("diagonal", 100, 0), ("chain", 64, 0), ("chain", 500, 0), ("scattered", 33, 0),
    ("scattered", 1, 0), ("wide", 900, 0), ("wide", 100, 0), ("grid", 700, 0), ("grid", 9000, 0), ("grid", 0, 3),
    ("direction_blocked", 150, 0), ("one", -5, 0), ("chain", -64, 0), ("scattered", -33, 0), ("wide", -100, 0),
    ("grid", -700, 0), ("grid", -1, 3), ("direction_blocked", -150, 0)])
@pytest.mark.parametrize("forward", [True, False], ids=["lower", "upper"])
@pytest.mark.parametrize("waves", [4, 12])
def test_layout_solves_bit_exactly(lib, kind, rows, cell, forward, waves):
    n, rp, ci, v = _matrix(kind)
    r = np.random.default_rng(9).standard_normal(n)
    x, info = np.zeros(n), np.zeros(8, np.int32)
    rc = lib.part_layout_run(n, rp.ctypes.data_as(ctypes.c_void_p), ci.ctypes.data_as(ctypes.c_void_p),
                             v.ctypes.data_as(ctypes.c_void_p), int(forward), rows, cell, waves,
                             r.ctypes.data_as(ctypes.c_void_p), x.ctypes.data_as(ctypes.c_void_p),
                             info.ctypes.data_as(ctypes.c_void_p))
    assert rc == 0
    if abs(rows) > 1:
        assert info[1] <= abs(rows)
    if kind == "wide" and rows == 100:
        assert info[4] > 200   # steps that close at their externals are among the cases
    assert np.array_equal(x, _reference(n, rp, ci, v, r, forward))


def test_grid_is_found_only_in_grid_numberings(lib):
    for kind, found in (("grid", True), ("chain", False), ("scattered", False), ("diagonal", False)):
        n, rp, ci, v = _matrix(kind)
        x, info = np.zeros(n), np.zeros(8, np.int32)
        rc = lib.part_layout_run(n, rp.ctypes.data_as(ctypes.c_void_p), ci.ctypes.data_as(ctypes.c_void_p),
                                 v.ctypes.data_as(ctypes.c_void_p), 1, 0, 3, 12,
                                 np.ones(n).ctypes.data_as(ctypes.c_void_p), x.ctypes.data_as(ctypes.c_void_p),
                                 info.ctypes.data_as(ctypes.c_void_p))
        assert (rc == 0) == found, (kind, rc)


def test_quotient_from_reciprocal_equals_division(lib):
    rng = np.random.default_rng(3)
    n = 4_000_000
    s = rng.standard_normal(n) * 2.0 ** rng.integers(-399, 399, n)
    d = rng.uniform(1.0, 2.0, n) * 2.0 ** rng.integers(-399, 398, n) * rng.choice([-1.0, 1.0], n)
    # mantissas next to powers of two and to each other, exact quotients, zeros of both signs
    s[:1000] = np.ldexp(1.0 + np.arange(1000) * 2.0 ** -52, 3)
    d[:1000] = np.ldexp(2.0 - (1 + np.arange(1000)[::-1]) * 2.0 ** -52, -5)
    s[1000:2000] = d[1000:2000] * 3.0
    s[2000:2010], s[2010:2020] = 0.0, -0.0
    keep = (np.abs(s) >= 2.0 ** -400) & (np.abs(s) <= 2.0 ** 400) | (s == 0.0)
    s, d = np.ascontiguousarray(s[keep]), np.ascontiguousarray(d[keep])
    q = np.zeros(len(s))
    lib.part_quotients(ctypes.c_long(len(s)), s.ctypes.data_as(ctypes.c_void_p), d.ctypes.data_as(ctypes.c_void_p),
                       q.ctypes.data_as(ctypes.c_void_p))
    assert np.array_equal(q.view(np.uint64), (s / d).view(np.uint64))


def test_oracle_plain_sweeps_agree_with_the_reference_loop():
    n, rp, ci, v = _matrix("direction_blocked")
    r = np.random.default_rng(1).standard_normal(n)
    x = _reference(n, rp, ci, v, r, True)
    keep = np.concatenate([ci[rp[i]:rp[i + 1]] <= i for i in range(n)])
    lrp = np.concatenate([[0], np.cumsum(np.add.reduceat(keep, rp[:-1]))]).astype(np.int32)
    assert np.array_equal(O.fr((lrp, ci[keep], v[keep]), r), x)


def test_host_failures_reach_the_caller(tmp_path):
    """No allocation and no thread start that fails ends the process (tests/cpp/part_alloc_main.cpp)."""
    exe = str(tmp_path / "part_alloc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-rdynamic", f"-I{ROOT}/sparsesolv_amd/csrc",
                    os.path.join(ROOT, "tests", "cpp", "part_alloc_main.cpp"), "-ldl", "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
    assert r.stdout.startswith("ok ") and int(r.stdout.split()[1]) > 50


def test_kernel_quotient_and_its_range(tmp_path):
    """The code the kernels run (ssgpu_quot.h), over the whole exponent range and at the edges of its own."""
    out = str(tmp_path / "libquot.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", "-shared", "-fPIC",
                    f"-I{ROOT}/sparsesolv_amd/csrc", os.path.join(ROOT, "tests", "cpp", "quot_main.cpp"), "-o", out],
                   check=True)
    lib = ctypes.CDLL(out)
    lib.quotients.restype = ctypes.c_long
    rng = np.random.default_rng(12)
    n = 2_000_000

    def values(k, lo, hi):
        return np.ldexp(rng.uniform(1.0, 2.0, k) * rng.choice([-1.0, 1.0], k), rng.integers(lo, hi, k))

    edges = np.array([2.0 ** e * m for e in (-401, -400, 399, 400) for m in (1.0, 1.0 + 2.0 ** -52, 2.0 - 2.0 ** -52)])
    special = np.array([0.0, -0.0, 5e-324, -5e-324, 2.0 ** -1022, 1.7976931348623157e308, np.inf, -np.inf, np.nan])
    s = np.concatenate([values(n, -1074, 1024), values(n, -400, 400), np.repeat(np.concatenate([edges, special]), 21)])
    d = np.concatenate([values(n, -1074, 1024), values(n, -400, 400), np.tile(np.concatenate([edges, special]), 21)])
    q = np.zeros(len(s))
    formed = lib.quotients(ctypes.c_long(len(s)), s.ctypes.data_as(ctypes.c_void_p),
                           d.ctypes.data_as(ctypes.c_void_p), q.ctypes.data_as(ctypes.c_void_p))
    assert n < formed < 2 * n
    with np.errstate(all="ignore"):
        want = s / d
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(q), nan)
    assert np.array_equal(q[~nan].view(np.uint64), want[~nan].view(np.uint64))


@pytest.mark.parametrize("kind,rows,cell", [("chain", 64, 0), ("scattered", 33, 0), ("wide", 100, 0), ("grid", 700, 0),
                                            ("grid", 0, 3), ("direction_blocked", -150, 0)])
@pytest.mark.parametrize("forward", [True, False], ids=["lower", "upper"])
def test_layout_of_eight_waves(lib, kind, rows, cell, forward):
    """The waves of real rows over 20 entries and of complex rows up to 20."""
    test_layout_solves_bit_exactly(lib, kind, rows, cell, forward, 8)
