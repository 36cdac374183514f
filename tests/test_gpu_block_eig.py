"""LOBPCG (plantfem_amd/csrc/eig.hip) at block widths that leave remainders in its kernels: one column,
exactly and one over the four columns that a product takes at once, and more than the 16 columns of the
middle form of the Rayleigh-Ritz update.  Reference: LAPACK on the reduced dense pencil."""

import numpy as np
import pytest
import scipy.linalg as sl

from test_modal import dense, modal_system


@pytest.mark.gpu
@pytest.mark.parametrize("nev", [1, 4, 5, 17])
def test_block_widths(ctx, nev):
    s, rp, ci, A, B, fixed = modal_system(ctx, (3, 3, 8), jitter=0.1)
    print("block width", nev, flush=True)
    tol = 1e-8
    lam, V = s.eig(num_eigen=nev, tol=tol)
    assert s.last_stats["status"] == 0
    n = rp.size - 1
    free = np.setdiff1d(np.arange(n), fixed - 1)
    Af, Bf = dense(rp, ci, A)[np.ix_(free, free)], dense(rp, ci, B)[np.ix_(free, free)]
    ref = sl.eigh(Af, Bf, eigvals_only=True)
    # a residual of tol |l| |B x| puts each value within tol |l| cond(B)^(1/2) of one of the pencil
    cond = np.linalg.cond(Bf)
    np.testing.assert_allclose(lam, ref[:nev], rtol=0, atol=2.0 * tol * ref[nev - 1] * np.sqrt(cond))
    np.testing.assert_allclose(V.T @ dense(rp, ci, B) @ V, np.eye(nev), atol=1e-7)
    assert np.all(V[fixed - 1] == 0.0)
