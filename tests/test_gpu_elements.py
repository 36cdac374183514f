"""The element-by-element stiffness product against the assembled CRS, and solves that use it.

The two sum the same terms in different orders, so a row differs by a few dozen roundings of its
absolute sum; the assembled element matrices also carry the cancellation of J = sum dN X, the
coordinates' size over the element's (64 eps (1 + max |X| / h) sum_j |a_ij| |x_j| in all)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")  # its HIP runtime starts before the library's

from plantfem_amd import _lib as L  # noqa: E402
from plantfem_amd import fem, workloads  # noqa: E402


def _apply(s, x):
    y = np.empty(s.n)
    L.check(L.load().pf_system_elem_apply(s.h, L.ptr(x, C.c_double), L.ptr(y, C.c_double)), "elem_apply")
    return y


def _jitter(nod, el, amount, seed):
    rng = np.random.default_rng(seed)
    h = np.ptp(nod, axis=0).max() / max(1, round(el.shape[0] ** (1 / 3)))
    return np.asfortranarray(nod + amount * h * rng.uniform(-1, 1, nod.shape)), el


def _permuted(nod, el, seed):
    rng = np.random.default_rng(seed)
    p = rng.permutation(nod.shape[0])  # new id of node i
    out = np.empty_like(nod, order="F")
    out[p] = nod
    return out, np.asfortranarray((p[el - 1] + 1).astype(np.int32)[rng.permutation(el.shape[0])])


def _wedge(nod, el):
    el = el.copy(order="F")
    el[::3, 3] = el[::3, 2]  # node listed twice
    el[::3, 7] = el[::3, 6]
    return nod, el


MESHES = {
    "one": lambda: fem.cube3d(1, 1, 1),
    "pair": lambda: fem.cube3d(2, 1, 1, 1.0, 2.0, 0.5),
    "odd": lambda: fem.cube3d(5, 7, 3, 1.0, 1.0, 1.0),
    "tile": lambda: fem.cube3d(8, 8, 4, 1.0, 1.0, 0.5),
    "past_tile": lambda: fem.cube3d(9, 8, 5),
    "needle": lambda: fem.cube3d(1, 1, 300, 0.01, 0.01, 3.0),
    "sheet": lambda: fem.cube3d(33, 1, 41, 1.0, 0.01, 1.0),
    "cylinder": lambda: fem.cylinder3d(10, 10, 9, 1.0, 1.0, 0.7),
    "leaf": lambda: fem.leaf3d(12, 2, 17, 0.12, 0.01, 0.2),
    "jittered": lambda: _jitter(*fem.cube3d(11, 10, 13), 0.2, 1),
    "permuted": lambda: _permuted(*_jitter(*fem.cube3d(12, 9, 10), 0.15, 2), 3),
    "wedges": lambda: _wedge(*fem.cube3d(7, 6, 5)),
    "unused_nodes": lambda: (np.asfortranarray(np.concatenate([fem.cube3d(4, 4, 4)[0], np.full((9, 3), np.nan)])),
                             fem.cube3d(4, 4, 4)[1]),
}


@pytest.mark.parametrize("jmode", [0, 1])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_product_matches_crs(name, jmode):
    nod, el = MESHES[name]()
    rng = np.random.default_rng(5)
    ne = el.shape[0]
    s = fem.FEMSolver()
    s.setDomain(fem.FEMDomain(nod, el))
    s.setCRS(DOF=3)
    s.setStiffness(1e7 * np.exp(rng.standard_normal(ne)), rng.uniform(0.0, 0.45, ne), jmode)
    x = rng.standard_normal(s.n)
    c = nod[el - 1]
    far = np.max(np.nanmax(np.abs(nod), axis=0) / np.ptp(c, axis=1).min(axis=0))
    # without fixes, with nonzero ones (unit rows, dropped columns), after a PointJacobi scaling,
    # with more fixes on the scaled matrix
    for step in range(4):
        if step == 1 or step == 3:
            s.fix(1, rng.integers(1, 3 * 8 + 1, 5).astype(np.int32) if step == 3 else
                  np.unique(rng.integers(1, s.n + 1, 1 + s.n // 7)).astype(np.int32), FixValue=0.25 * step)
        if step == 2:
            s.solve(preconditioning="PointJacobi", jacobi_solve=False)
        y = _apply(s, x)
        A = s.getCRS().to_scipy()
        B = abs(A)
        assert np.all(np.isfinite(A.data))
        assert np.all(np.abs(y - A @ x) <= 64 * np.finfo(float).eps * (1 + far) * (B @ np.abs(x))), (name, step)


def test_same_on_every_run():
    nod, el = MESHES["permuted"]()
    s = fem.FEMSolver()
    s.setDomain(fem.FEMDomain(nod, el))
    s.setCRS(DOF=3)
    s.setStiffness(np.full(el.shape[0], 1e7), np.full(el.shape[0], 0.3))
    x = np.random.default_rng(1).standard_normal(s.n)
    y = _apply(s, x)
    for _ in range(3):
        assert np.array_equal(y, _apply(s, x))


def test_only_for_a_stiffness():
    """Values from anything but the stiffness assembly are never replaced by it."""
    nod, el = fem.cube3d(3, 3, 3)
    s = fem.FEMSolver()
    s.setDomain(fem.FEMDomain(nod, el))
    s.setCRS(DOF=3)
    x = np.ones(s.n)

    def refused():
        with pytest.raises(Exception):
            _apply(s, x)

    refused()  # zero values
    E, nu = np.full(27, 1e7), np.full(27, 0.3)
    s.setStiffness(E, nu)
    _apply(s, x)
    s.setMatrix(1, 1, 3, np.eye(24))
    s._flush()
    refused()
    s.setStiffness(E, nu)
    _apply(s, x)
    s.setMassMatrix(1.0)
    refused()
    s.setStiffness(E, nu)
    s.zeros()
    refused()
    s.setStiffness(E, nu)
    s.setCRS(CRS=s.getCRS())
    refused()
    loose = np.arange(1, 8 * 5000 + 1, dtype=np.int32).reshape(5000, 8)  # no shared node
    s = fem.FEMSolver()
    s.setDomain(fem.FEMDomain(np.random.default_rng(0).uniform(size=(40000, 3)), loose))
    s.setCRS(DOF=3)
    s.setStiffness(np.full(5000, 1e7), np.full(5000, 0.3))
    with pytest.raises(Exception):
        _apply(s, np.ones(s.n))


@pytest.mark.parametrize("kw", [{"precision": 64}, {"precision": 48}, {"precision": 32},
                                {"precision": 64, "preconditioning": "PointJacobi"},
                                {"precision": 48, "preconditioning": "PointJacobi"}])
@pytest.mark.parametrize("mesh", ["box", "cylinder"])
def test_solve(mesh, kw):
    """Solves above the size at which the product is taken agree with the CRS-row solves (both to a
    relative residual of 1e-10, an error of about 1e-8 on these systems)."""
    nod, el = fem.cube3d(41, 29, 37) if mesh == "box" else fem.cylinder3d(18, 18, 30, 1.0, 1.0, 1.6)
    rng = np.random.default_rng(3)
    ne = el.shape[0]
    E, nu = 1e7 * np.exp(0.5 * rng.standard_normal(ne)), rng.uniform(0.25, 0.35, ne)
    base = np.nonzero(nod[:, 2] <= nod[:, 2].min())[0]
    ids = (3 * base[:, None] + np.arange(1, 4)).ravel().astype(np.int32)
    z = nod[:, 2].max()
    out = []
    for extra in ({}, {"spmv_kind": 1}):
        s = fem.FEMSolver()
        s.setDomain(fem.FEMDomain(nod, el))
        s.setCRS(DOF=3)
        s.setStiffness(E, nu)
        s.addTraction([-1e300, 1e300, -1e300, 1e300, z - 1e-9, z + 1e-9], -1e4)
        s.fix(1, ids, FixValue=0.0)
        s.fix(1, np.array([3 * base[0] + 3], np.int32), FixValue=1e-4)  # a nonzero support displacement
        s.relative_er = 1e-10
        k = dict(kw)
        if k["precision"] != 64:
            k["target_relres"] = 1e-10
        out.append(s.solve(stop_mode=1, **k, **extra))
        assert s.last_stats["status"] == 0 and s.last_stats["true_relres"] < 2e-10
        assert s.last_stats["spmv_kind_used"] == (1 if extra else 5)
    assert np.linalg.norm(out[0] - out[1]) <= 1e-7 * np.linalg.norm(out[1])


def _system(nod, el, seed=0):
    rng = np.random.default_rng(seed)
    s = fem.FEMSolver()
    s.setDomain(fem.FEMDomain(nod, el))
    s.setCRS(DOF=3)
    s.setStiffness(1e7 * np.exp(0.3 * rng.standard_normal(el.shape[0])), np.full(el.shape[0], 0.3))
    return s


@pytest.mark.parametrize("other", ["same", "larger", "smaller"])
def test_mesh_replaced_under_the_matrix(other):
    """A new mesh leaves the CRS as it was: products with it are those of the CRS, never of the new mesh."""
    nod, el = fem.cube3d(6, 6, 6)
    s = _system(nod, el)
    x = np.random.default_rng(1).standard_normal(s.n)
    y = _apply(s, x)
    new = {"same": (np.asfortranarray(nod * [1.0, 2.0, 0.5]), el), "larger": fem.cube3d(9, 9, 9),
           "smaller": fem.cube3d(2, 2, 2)}[other]
    s.setDomain(fem.FEMDomain(*new))
    with pytest.raises(L.PFError):
        _apply(s, x)
    A = s.getCRS().to_scipy()
    assert np.all(np.abs(A @ x - y) <= 1e-12 * (abs(A) @ np.abs(x)))
    s.setCRS(DOF=3)  # and with a stiffness of the new mesh the product is back
    s.setStiffness(np.full(new[1].shape[0], 1e7), np.full(new[1].shape[0], 0.3))
    x = np.random.default_rng(2).standard_normal(s.n)
    A = s.getCRS().to_scipy()
    assert np.all(np.abs(_apply(s, x) - A @ x) <= 1e-12 * (abs(A) @ np.abs(x)))


@pytest.mark.parametrize("precision", [64, 48])
def test_solve_after_the_mesh_moved(precision):
    """The solve is that of the stored CRS when the mesh was replaced after the assembly."""
    nod, el = fem.cube3d(29, 28, 27)  # 73,080 rows: the element form in its range
    s = _system(nod, el)
    s.addTraction([-1e300, 1e300, -1e300, 1e300, 1 - 1e-9, 1 + 1e-9], -1e4)
    base = np.nonzero(nod[:, 2] == 0)[0]
    s.fix(1, (3 * base[:, None] + np.arange(1, 4)).ravel().astype(np.int32), FixValue=0.0)
    s.setDomain(fem.FEMDomain(np.asfortranarray(nod * [1.0, 3.0, 0.5]), el))
    s.relative_er = 1e-10
    s.solve(precision=precision, stop_mode=1, target_relres=1e-10)
    assert s.last_stats["status"] == 0 and s.last_stats["true_relres"] < 2e-10
    assert s.last_stats["spmv_kind_used"] != 5


def _array(ptr, count):
    """A torch tensor over device memory (float64)."""
    class Mem:
        __cuda_array_interface__ = {"shape": (count,), "typestr": "<f8", "version": 2,
                                    "data": (C.cast(ptr, C.c_void_p).value, False)}

    return torch.as_tensor(Mem(), device="cuda")


@pytest.mark.parametrize("precision", [64, 48])
def test_writes_through_an_earlier_view(precision):
    """Values and coordinates written through a view that was taken before the assembly count."""
    nod, el = fem.cube3d(29, 28, 27)
    s = _system(nod, el)
    _apply(s, np.ones(s.n))  # the tiles of the mesh as it is
    v = L.SystemView()
    L.check(L.load().pf_system_view_get(s.h, C.byref(v)), "view")
    top = [-1e300, 1e300, -1e300, 1e300, 1 - 1e-9, 1 + 1e-9]
    base = np.nonzero(nod[:, 2] == 0)[0]
    ids = (3 * base[:, None] + np.arange(1, 4)).ravel().astype(np.int32)
    s.relative_er = 1e-10
    s.addTraction(top, -1e4)
    s.fix(1, ids, FixValue=0.0)
    _array(v.nodcoord, 3 * nod.shape[0])[: nod.shape[0]] *= 2.0  # x of every node
    torch.cuda.synchronize()
    s.setStiffness()
    _array(v.val, int(v.nnz)).mul_(3.0)
    torch.cuda.synchronize()
    with pytest.raises(L.PFError):
        _apply(s, np.ones(s.n))
    s.solve(precision=precision, stop_mode=1, target_relres=1e-10)
    assert s.last_stats["status"] == 0 and s.last_stats["true_relres"] < 2e-10
    assert s.last_stats["spmv_kind_used"] != 5
    # the pointers end with the CRS; the tiles are then those of the moved nodes
    s.setCRS(DOF=3)
    s.setStiffness()
    x = np.random.default_rng(2).standard_normal(s.n)
    A = s.getCRS().to_scipy()
    assert np.all(np.abs(_apply(s, x) - A @ x) <= 1e-11 * (abs(A) @ np.abs(x)))


@pytest.mark.parametrize("kw", [{"inner_max": 1}, {"inner_max": 2}, {"inner_max": 6}, {"inner_max": 7}, {"inner_max": 33},
                                {"inner_tol": 0.5}, {"inner_tol": 0.7}, {"inner_tol": 0.95}])
@pytest.mark.parametrize("precision,dims", [(32, (9, 8, 7)), (48, (9, 8, 7)), (48, (29, 28, 27))])
def test_replacement_intervals(precision, dims, kw):
    """Residual replacements asked for after every few iterations are done as asked: no iteration is run
    between the request and the replacement, whatever the interval at which they are looked for."""
    nod, el = fem.cube3d(*dims)
    s = _system(nod, el)
    s.addTraction([-1e300, 1e300, -1e300, 1e300, 1 - 1e-9, 1 + 1e-9], -1e4)
    base = np.nonzero(nod[:, 2] == 0)[0]
    s.fix(1, (3 * base[:, None] + np.arange(1, 4)).ravel().astype(np.int32), FixValue=0.0)
    s.itrmax = 66
    s.solve(precision=precision, target_relres=1e-30, raise_on_breakdown=False, **kw)
    st = s.last_stats
    assert st["iterations"] <= 66
    # products of the assembled matrix where the replacements, which use it, are most of the work
    often = kw.get("inner_max", 9) < 4 or kw.get("inner_tol", 0) > 0.8
    assert st["spmv_kind_used"] == (5 if s.n >= 40000 and not often else 2)
    if "inner_max" in kw:  # one at least every inner_max iterations (the last iteration asks for none)
        assert st["outer_iterations"] >= (st["iterations"] - 1) // kw["inner_max"]
