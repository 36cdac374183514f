"""Small FP64 solves, whose iterations run in one kernel (the automatic choice), against the CRS-row
launches (spmv_kind 1) and dense solutions.

Both stop at |r| < 1e-12 |b| on matrices with a condition number below 100, so the solutions lie
within 100 * 1e-12 of the exact one, 1e-9 with room."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from plantfem_amd import _lib as L  # noqa: E402
from plantfem_amd.fem import FEMDomain, FEMSolver, bicgstab_crs, cube3d  # noqa: E402


def _one_kernel():
    return L.default_context().forms()["one_kernel"]


def _crs(rows):
    """1-based CRS of a list of {column: value}, columns in the order given."""
    rp = np.cumsum([1] + [len(r) for r in rows]).astype(np.int64)
    ci = np.array([c + 1 for r in rows for c in r], np.int32)
    return rp, ci, np.array([v for r in rows for v in r.values()], float)


def _matrix(kind, n, seed=0):
    rng = np.random.default_rng(seed)
    rows = []
    for i in range(n):
        if kind == "tridiagonal":
            cols = [c for c in (i + 1, i - 1) if 0 <= c < n]
        elif kind == "ragged":  # 0 to 60 neighbours, some rows of one entry
            cols = [c for c in rng.integers(i - 40, i + 41, rng.integers(0, 61)) if 0 <= c < n and c != i]
        elif kind == "long":  # a few rows of hundreds of entries among short ones
            m = 700 if i % 97 == 5 else 4
            cols = [c for c in rng.integers(max(0, i - 800), min(n, i + 800), m) if c != i]
        else:  # scattered: from 8000 rows on more distinct columns per workgroup than it stages
            cols = [c for c in rng.integers(0, n, 90) if c != i]
        row = {int(c): float(rng.uniform(-1, 1)) for c in cols}
        row[i] = 1.5 * sum(abs(v) for v in row.values()) + 1.0
        rows.append(row)
    return rows


def _dense(rows):
    A = np.zeros((len(rows), len(rows)))
    for i, r in enumerate(rows):
        A[i, list(r)] = list(r.values())
    return A


@pytest.mark.parametrize("kind,n", [("tridiagonal", 2), ("tridiagonal", 63), ("tridiagonal", 64), ("tridiagonal", 511), ("tridiagonal", 513),
                                    ("tridiagonal", 4000), ("ragged", 64), ("ragged", 513), ("ragged", 3000),
                                    ("long", 3000), ("scattered", 4100)])
@pytest.mark.parametrize("x0", [False, True])
def test_general_matrices(kind, n, x0):
    rows = _matrix(kind, n)
    A = _dense(rows)
    rng = np.random.default_rng(1)
    b = rng.standard_normal(n)
    start = rng.standard_normal(n) if x0 else None
    crs = _crs(rows)
    ref = np.linalg.solve(A, b)
    for k in (0, 1):
        x, st = bicgstab_crs(*crs, b, x0=start, stop_mode=1, relative_er=1e-12, spmv_kind=k)
        assert st["status"] == 0 and st["true_relres"] < 1e-11
        assert np.linalg.norm(x - ref) <= 1e-9 * np.linalg.norm(ref), (k, st)
        # launches below 64 rows, and where a workgroup's 2048 entries are more than 512 rows (three per row)
        assert _one_kernel() == (k == 0 and n >= 64 and not (kind == "tridiagonal" and n > 512))


def test_too_many_columns():
    """More distinct columns per workgroup than it stages: the launches run."""
    n = 8000
    crs = _crs(_matrix("scattered", n))
    b = np.random.default_rng(4).standard_normal(n)
    out = []
    for k in (0, 1):
        x, st = bicgstab_crs(*crs, b, stop_mode=1, relative_er=1e-12, spmv_kind=k)
        assert st["status"] == 0 and st["true_relres"] < 1e-11 and _one_kernel() == 0
        out.append(x)
    assert np.linalg.norm(out[0] - out[1]) <= 1e-9 * np.linalg.norm(out[1])


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_stop_rules_and_counts(mode):
    rows = _matrix("ragged", 2000)
    crs = _crs(rows)
    b = np.random.default_rng(2).standard_normal(2000)
    kw = {"stop_mode": mode, "relative_er": 1e-10, "er0": 1e-20 if mode == 2 else 1e-300}
    x0, s0 = bicgstab_crs(*crs, b, spmv_kind=0, **kw)
    assert _one_kernel() == 1
    x1, s1 = bicgstab_crs(*crs, b, spmv_kind=1, **kw)
    assert s0["status"] == s1["status"] == 0 and s0["iterations"] == s1["iterations"]
    assert np.linalg.norm(x0 - x1) <= 1e-9 * np.linalg.norm(x1)
    for m in (1, 2, 7):  # iterates of a few steps differ by rounding only
        x0, s0 = bicgstab_crs(*crs, b, spmv_kind=0, itrmax=m, stop_mode=1, relative_er=1e-30)
        x1, s1 = bicgstab_crs(*crs, b, spmv_kind=1, itrmax=m, stop_mode=1, relative_er=1e-30)
        assert s0["iterations"] == s1["iterations"] == m and s0["status"] == s1["status"] == 3
        assert np.linalg.norm(x0 - x1) <= 1e-12 * np.linalg.norm(x1)


def test_empty_rows_and_zero_rhs():
    rows = _matrix("ragged", 900)
    for i in range(0, 900, 7):
        rows[i] = {}
    for r in rows:
        for c in [c for c in r if c % 7 == 0]:
            del r[c]
    keep = np.arange(900) % 7 != 0
    b = np.where(keep, np.random.default_rng(3).standard_normal(900), 0.0)
    x, st = bicgstab_crs(*_crs(rows), b, stop_mode=1, relative_er=1e-12)
    assert _one_kernel() == 1
    ref = np.zeros(900)
    ref[keep] = np.linalg.solve(_dense(rows)[np.ix_(keep, keep)], b[keep])
    assert st["status"] == 0 and np.linalg.norm(x - ref) <= 1e-9 * np.linalg.norm(ref)
    x0, s0 = bicgstab_crs(*_crs(rows), np.zeros(900), spmv_kind=0)
    x1, s1 = bicgstab_crs(*_crs(rows), np.zeros(900), spmv_kind=1)
    assert s0["status"] == s1["status"] and np.array_equal(x0, x1, equal_nan=True)


def test_breakdown_and_nan():
    """A = c I: e = 0 and v.v = 0 in the first iteration, before x moves; a NaN load ends."""
    for n in (1, 100, 5000):
        rows = [{i: 2.0} for i in range(n)]
        for k in (0, 1):
            x, st = bicgstab_crs(*_crs(rows), np.ones(n), spmv_kind=k, er0=0.0, relative_er=0.0)
            assert st["status"] == 1 and st["iterations"] == 1 and not x.any(), (k, st)
            assert _one_kernel() == (k == 0 and n == 100)  # of 5000 rows with one entry each a workgroup gets 2048
        b = np.ones(n)
        b[n // 2] = np.nan
        x, st = bicgstab_crs(*_crs(rows), b, stop_mode=1, relative_er=1e-10, itrmax=50)
        assert st["status"] != 0


@pytest.mark.parametrize("dims", [(4, 3, 5), (9, 9, 9), (23, 20, 22)])
def test_same_on_every_run(dims):
    nod, el = cube3d(*dims)
    s = FEMSolver()
    s.setDomain(FEMDomain(nod, el))
    out = []
    for _ in range(3):
        s.setCRS(DOF=3)
        s.setStiffness(np.full(el.shape[0], 1e7), np.full(el.shape[0], 0.3))
        s.addTraction([-1e300, 1e300, -1e300, 1e300, 1 - 1e-9, 1 + 1e-9], -1e4)
        base = np.nonzero(nod[:, 2] == 0)[0]
        s.fix(1, (3 * base[:, None] + np.arange(1, 4)).ravel().astype(np.int32), FixValue=0.0)
        out.append(s.solve())
        assert _one_kernel() == 1
        assert s.last_stats["status"] == 0 and s.last_stats["true_relres"] < 1e-8
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])
