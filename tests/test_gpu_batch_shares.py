"""Batched BiCGSTAB with meshes that several workgroups share (plantfem_amd/csrc/batch.hip), in FP64 and
mixed precision, on the blocked layout (shares end at 64-node slices, the last one short) and on CRS
rows, beside meshes of one workgroup.  Each mesh's solution is checked through the residual of its own
eliminated system, recomputed on the CPU from the oracle's matrix."""

import numpy as np
import pytest

from plantfem_amd import batch as B
from test_direct import organ_system, relres, rounding_floor, to_scipy

REL = 1e-9


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("tune", [None, {"layout": 0, "sub": 16, "block": 256, "blocks_per_cu": 0},
                                  {"layout": 1, "sub": 64, "block": 1024, "blocks_per_cu": 1}])
def test_shared_meshes(ctx, precision, tune):
    rng = np.random.default_rng(11)
    organs = [B.block(n, rng) for n in (3, 13, 10, 5, 11)]  # 8232 rows: up to 4 shares; 3993 rows: one
    u = B.union(organs)
    s = B.build_solver(u, ctx)
    s.relative_er = REL
    print("shared batch", precision, tune, flush=True)
    for again in range(2):  # the second solve starts from the first one's meeting counters
        x, st = s.solveBatch(precision=precision, tune=tune, stop_mode=1, target_relres=REL)
        assert ctx.forms()["batch_shares"] > 1
    s.close()
    for m, o in enumerate(organs):
        rp, ci, val, rhs = organ_system(o)
        A, xm = to_scipy(rp, ci, val), x[u.dof_range(m)]
        res = relres(A, xm, rhs)
        assert st["status"][m] == 0
        # FP64 stops on the recursive residual, which leaves the true one by rounding only
        assert res <= REL * (1.0 if precision == 32 else 1.5) + rounding_floor(A, xm, rhs)
        assert abs(res - st["true_relres"][m]) <= 10.0 * rounding_floor(A, xm, rhs)


@pytest.mark.gpu
def test_one_shared_mesh_matches_the_single_solver(ctx):
    """A batch of one mesh (the first rule's largest shares) against the oracle's recurrence."""
    rng = np.random.default_rng(12)
    o = B.block(12, rng)
    u = B.union([o])
    s = B.build_solver(u, ctx)
    s.relative_er = REL
    print("one shared mesh", flush=True)
    x, st = s.solveBatch(stop_mode=1)
    assert ctx.forms()["batch_shares"] > 1
    s.close()
    rp, ci, val, rhs = organ_system(o)
    A = to_scipy(rp, ci, val)
    assert st["status"][0] == 0
    assert relres(A, x, rhs) <= 1.5 * REL + rounding_floor(A, x, rhs)


@pytest.mark.gpu
@pytest.mark.parametrize("per_cu", [0, 1, 2])
def test_workgroups_per_cu_with_shares(ctx, per_cu):
    """The caller's number of workgroups per CU counts with shared meshes too; left open it is one."""
    rng = np.random.default_rng(13)
    u = B.union([B.block(13, rng)] + [B.block(2, rng) for _ in range(300)])
    s = B.build_solver(u, ctx)
    s.relative_er = REL
    print("workgroups per CU", per_cu, flush=True)
    x, st = s.solveBatch(tune={"layout": 1, "sub": 64, "block": 256, "blocks_per_cu": per_cu}, stop_mode=1)
    s.close()
    assert not st["status"].any() and np.all(st["true_relres"] <= 1.5 * REL) and ctx.forms()["batch_shares"] > 1
    assert (st["workgroup"].max() >= 256) == (per_cu == 2)  # 256 CUs
