"""Solves whose workgroups wait for each other, where such launches are refused or a wait gives up: the same
systems by launches (plantfem_amd/csrc/bicgstab.hip) and with whole meshes (batch.hip, direct.hip)."""

import numpy as np
import pytest
import scipy.linalg as sl

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")  # its HIP runtime starts before the library's

from plantfem_amd import _lib as L  # noqa: E402
from plantfem_amd import batch as B  # noqa: E402
from plantfem_amd.fem import bicgstab_crs  # noqa: E402
from test_direct import organ_system, relres, rounding_floor, to_scipy  # noqa: E402
from test_gpu_direct_bands import EPS, band_system, solver  # noqa: E402
from test_gpu_one_kernel import _crs, _matrix  # noqa: E402

REL = 1e-9


@pytest.fixture
def alone():
    c = L.Context(0)
    c.together(False)
    yield c
    c.close()


@pytest.mark.parametrize("x0", [False, True])
def test_one_kernel_refused(alone, x0):
    crs = _crs(_matrix("ragged", 3000))
    rng = np.random.default_rng(1)
    b = rng.standard_normal(3000)
    start = rng.standard_normal(3000) if x0 else None
    kw = {"x0": start, "ctx": alone, "stop_mode": 1, "relative_er": 1e-12}
    x, st = bicgstab_crs(*crs, b, **kw)
    assert alone.forms()["one_kernel"] == 0 and st["status"] == 0
    y, sy = bicgstab_crs(*crs, b, spmv_kind=1, **kw)  # the same launches
    assert np.array_equal(x, y) and st["iterations"] == sy["iterations"]


@pytest.mark.parametrize("precision", [64, 32])
def test_batch_shares_refused(alone, precision):
    rng = np.random.default_rng(11)
    organs = [B.block(n, rng) for n in (3, 13, 10, 5, 11)]
    u = B.union(organs)
    s = B.build_solver(u, alone)
    s.relative_er = REL
    print("whole meshes", precision, flush=True)
    out = []
    for _ in range(3):  # the first solve is refused, the others start with whole meshes (and a graph)
        x, st = s.solveBatch(precision=precision, stop_mode=1, target_relres=REL)
        assert alone.forms()["batch_shares"] == 1
        out.append(x)
    s.close()
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])
    for m, o in enumerate(organs):
        rp, ci, val, rhs = organ_system(o)
        A, xm = to_scipy(rp, ci, val), out[0][u.dof_range(m)]
        assert st["status"][m] == 0
        assert relres(A, xm, rhs) <= REL * (1.0 if precision == 32 else 1.5) + rounding_floor(A, xm, rhs)


@pytest.mark.parametrize("bad", [None, 700])
def test_direct_shares_refused(alone, bad):
    n, kd = 1499, 300
    lower, rp, ci, val, rhs = band_system(n, kd, 3)
    print("whole mesh", bad, flush=True)
    if bad is not None:
        v = val.copy()
        v[rp[bad] - 1 + min(bad, kd)] *= -1.0  # the diagonal entry
        s = solver(alone, rp, ci, v, rhs)
        with pytest.raises(L.PFError) as e:
            s.solve(algorithm="GaussJordan")
        assert e.value.code == L.PF_NOT_SPD
    else:
        s = solver(alone, rp, ci, val, rhs)
        ref = sl.solveh_banded(lower, rhs, lower=True)
        for _ in range(2):  # the second solve keeps the factor
            x = s.solve(algorithm="GaussJordan", refine=0)
            assert np.linalg.norm(x - ref) <= 2 * 4 * 20 * (kd + 1) * EPS * np.linalg.norm(ref)
    assert alone.forms()["direct_shares"] == 1
    s.close()


@pytest.fixture
def impatient():
    """Every wait ends after one poll, so that workgroups give up where another is not there yet."""
    c = L.Context(0)
    c.together(True, polls=1)
    yield c
    c.close()


@pytest.mark.parametrize("bad", [None, 700, 1498])
def test_direct_shares_that_give_up(impatient, bad):
    n, kd = 1499, 300
    lower, rp, ci, val, rhs = band_system(n, kd, 3)
    print("shares give up", bad, flush=True)
    if bad is not None:
        v = val.copy()
        v[rp[bad] - 1 + min(bad, kd)] *= -1.0  # the diagonal entry
        s = solver(impatient, rp, ci, v, rhs)
        with pytest.raises(L.PFError) as e:
            s.solve(algorithm="GaussJordan")
        assert e.value.code == L.PF_NOT_SPD
    else:
        s = solver(impatient, rp, ci, val, rhs)
        ref = sl.solveh_banded(lower, rhs, lower=True)
        for _ in range(2):  # the second solve keeps the factor
            x = s.solve(algorithm="GaussJordan", refine=0)
            assert np.linalg.norm(x - ref) <= 2 * 4 * 20 * (kd + 1) * EPS * np.linalg.norm(ref)
    assert impatient.forms()["direct_shares"] == 1
    s.close()


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("tune", [None, {"layout": 0, "sub": 16, "block": 256, "blocks_per_cu": 0}])
def test_batch_shares_that_give_up(impatient, alone, precision, tune):
    out = []
    for c in (impatient, alone):
        rng = np.random.default_rng(11)
        u = B.union([B.block(n, rng) for n in (3, 13, 10, 5, 11)])
        s = B.build_solver(u, c)
        s.relative_er = REL
        print("shares give up", precision, tune, flush=True)
        for _ in range(2):
            x, st = s.solveBatch(precision=precision, tune=tune, stop_mode=1, target_relres=REL)
            assert not st["status"].any() and c.forms()["batch_shares"] == 1
            out.append(x)
        s.close()
    for x in out[:-1]:  # the solve that was done again is the one without shares
        assert np.array_equal(x, out[-1])


@pytest.mark.parametrize("x0", [False, True])
def test_one_kernel_that_gives_up(impatient, alone, x0):
    crs = _crs(_matrix("ragged", 3000))
    rng = np.random.default_rng(1)
    b = rng.standard_normal(3000)
    kw = {"x0": rng.standard_normal(3000) if x0 else None, "stop_mode": 1, "relative_er": 1e-12}
    print("one kernel gives up", x0, flush=True)
    x, st = bicgstab_crs(*crs, b, ctx=impatient, **kw)
    y, sy = bicgstab_crs(*crs, b, ctx=alone, **kw)
    assert impatient.forms()["one_kernel"] == 0 and st["status"] == 0
    assert np.array_equal(x, y) and st["iterations"] == sy["iterations"]
    impatient.together(True)
    ran = []
    for _ in range(17):  # launches at once for a while, then the one kernel again
        x, st = bicgstab_crs(*crs, b, ctx=impatient, **kw)
        ran.append(impatient.forms()["one_kernel"])
        assert st["status"] == 0 and np.linalg.norm(x - y) <= 1e-9 * np.linalg.norm(y)
    assert ran == [0] * 16 + [1]


def test_one_workgroup_waits_for_none(alone):
    """A system that one workgroup holds needs no such launch and takes its kernel all the same."""
    crs = _crs(_matrix("tridiagonal", 300))
    b = np.random.default_rng(2).standard_normal(300)
    x, st = bicgstab_crs(*crs, b, ctx=alone, stop_mode=1, relative_er=1e-12)
    assert alone.forms()["one_kernel"] == 1 and st["status"] == 0 and st["true_relres"] < 1e-11


def test_threads():
    """Contexts in threads of their own, each with solves whose workgroups wait for each other: the launches
    take turns, and every result is that of a solve alone."""
    import threading
    crs = _crs(_matrix("ragged", 3000))
    rng = np.random.default_rng(1)
    b = rng.standard_normal(3000)
    lower, rp, ci, val, rhs = band_system(1499, 300, 3)
    u = B.union([B.block(n, rng) for n in (3, 13, 10)])

    def one(c, out):
        for _ in range(20):
            out.append((bicgstab_crs(*crs, b, ctx=c, stop_mode=1, relative_er=1e-12)[0], c.forms()["one_kernel"]))

    def direct(c, out):
        s = solver(c, rp, ci, val, rhs)
        for _ in range(10):
            s.setDirectKernel(True)  # drops the factor
            out.append((s.solve(algorithm="GaussJordan", refine=0), c.forms()["direct_shares"]))
        s.close()

    def shares(c, out):
        s = B.build_solver(u, c)
        s.relative_er = REL
        for _ in range(4):
            out.append((s.solveBatch(stop_mode=1)[0], c.forms()["batch_shares"]))
        s.close()

    print("threads", flush=True)
    work = [one, direct, shares]
    ctxs = [L.Context(0) for _ in range(2 * len(work))]
    logs = [[] for _ in ctxs]
    for f, c, out in zip(work, ctxs, logs):  # alone
        f(c, out)
    threads = [threading.Thread(target=f, args=(c, out)) for f, c, out in zip(work, ctxs[3:], logs[3:])]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for c in ctxs:
        c.close()
    for first, second in zip(logs[:3], logs[3:]):
        assert len(first) == len(second)
        for x, form in first + second:
            assert np.array_equal(x, first[0][0]) and form == first[0][1]
