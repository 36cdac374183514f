"""The banded direct solve (plantfem_amd/csrc/direct.hip) at the edges of its variants: half bandwidths
around 256, 512 and 1024 (the forms of the triangular solves and of the factorization's tiles; above
1024 the solves by blocks of 16), orders that leave a padded block, one block, meshes that several
workgroups factor in shares, and a non-positive pivot in such a mesh.  Reference: LAPACK's banded
Cholesky (scipy.linalg.solveh_banded)."""

import numpy as np
import pytest
import scipy.linalg as sl

EPS = np.finfo(float).eps


def band_system(n, kd, seed):
    """Random symmetric band matrix, normal entries off the diagonal (spectral radius about
    2 sqrt(2 kd)) and 2 kd + 3 on it; returns (lower band, row_ptr, col_idx, values, rhs)."""
    rng = np.random.default_rng(seed)
    lower = np.zeros((kd + 1, n))
    lower[0] = 2 * kd + 3
    for d in range(1, kd + 1):
        lower[d, : n - d] = rng.standard_normal(max(n - d, 0)) if d < n else 0.0
    i = np.arange(n)[:, None]
    j = i + np.arange(-kd, kd + 1)[None, :]
    inside = (j >= 0) & (j < n)
    jj = np.clip(j, 0, n - 1)
    val = lower[np.abs(i - jj), np.minimum(i, jj)]
    rp = np.concatenate([[1], 1 + np.cumsum(inside.sum(1))]).astype(np.int64)
    return lower, rp, (jj[inside] + 1).astype(np.int32), val[inside], rng.standard_normal(n)


def solver(ctx, rp, ci, val, rhs):
    from plantfem_amd.fem import CRS, FEMSolver
    s = FEMSolver(ctx)
    s.setCRS(CRS=CRS(rp, ci, val))
    s.setRHS(rhs)
    return s


@pytest.mark.gpu
@pytest.mark.parametrize("mfma", [True, False])
@pytest.mark.parametrize("n,kd", [(1, 0), (31, 5), (33, 32), (300, 224), (500, 256), (1001, 257), (1200, 480),
                                  (1100, 512), (1250, 513), (2100, 736), (2000, 737), (2200, 1024), (1500, 1100)])
def test_band_solve(ctx, n, kd, mfma):
    kd = min(kd, n - 1)
    print("band", n, kd, mfma, flush=True)
    lower, rp, ci, val, rhs = band_system(n, kd, n + kd)
    s = solver(ctx, rp, ci, val, rhs)
    s.setDirectKernel(mfma)
    x = s.solve(algorithm="GaussJordan", refine=0)
    assert (ctx.forms()["direct_shares"] > 1) == (n > 32 and kd <= 1024)
    assert s.directInfo()["bandwidth"] <= kd
    s.close()
    ref = sl.solveh_banded(lower, rhs, lower=True)
    # both solves are backward stable: each is off by at most a small multiple of (kd + 1) eps times
    # the condition number, which is below 20 for these spectra
    assert np.linalg.norm(x - ref) <= 2 * 4 * 20 * (kd + 1) * EPS * np.linalg.norm(ref)


@pytest.mark.gpu
@pytest.mark.parametrize("row", [0, 700, 1498])
def test_bad_pivot_in_a_shared_mesh(ctx, row):
    from plantfem_amd import _lib as L
    n, kd = 1499, 300
    lower, rp, ci, val, rhs = band_system(n, kd, 3)
    print("bad pivot", row, flush=True)
    bad = val.copy()
    bad[rp[row] - 1 + min(row, kd)] *= -1.0  # the diagonal entry
    s = solver(ctx, rp, ci, bad, rhs)
    with pytest.raises(L.PFError) as e:
        s.solve(algorithm="GaussJordan")
    assert e.value.code == L.PF_NOT_SPD and ctx.forms()["direct_shares"] > 1
    from plantfem_amd.fem import CRS
    s.setCRS(CRS=CRS(rp, ci, val))
    s.setRHS(rhs)
    x = s.solve(algorithm="GaussJordan", refine=0)
    s.close()
    ref = sl.solveh_banded(lower, rhs, lower=True)
    assert np.linalg.norm(x - ref) <= 2 * 4 * 20 * (kd + 1) * EPS * np.linalg.norm(ref)


@pytest.mark.gpu
@pytest.mark.parametrize("row", [0, 800, 1499])
@pytest.mark.parametrize("mfma", [True, False])
def test_bad_pivot_in_a_wide_band(ctx, row, mfma):
    """Above half bandwidth 1024 one workgroup factors and solves the mesh and has no progress to publish."""
    from plantfem_amd import _lib as L
    n, kd = 1500, 1100
    lower, rp, ci, val, rhs = band_system(n, kd, 4)
    print("bad pivot, wide", row, mfma, flush=True)
    bad = val.copy()
    bad[rp[row] - 1 + min(row, kd)] *= -1.0  # the diagonal entry
    s = solver(ctx, rp, ci, bad, rhs)
    s.setDirectKernel(mfma)
    with pytest.raises(L.PFError) as e:
        s.solve(algorithm="GaussJordan")
    assert e.value.code == L.PF_NOT_SPD and ctx.forms()["direct_shares"] == 1
    s.close()
