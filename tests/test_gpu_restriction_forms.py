"""The restriction's two forms: a thread per DOF, and per node on 75,000 coarse nodes x vectors and
more.  Both sum a DOF's fine partners in the same order with weights that are powers of two."""
import numpy as np
import pytest

from topopt3d_amd import configs

pytestmark = pytest.mark.gpu


# level 1 has 9,537 nodes on both: 7 vectors are below the line, 8 above it; the second mesh has
# levels with an even node count, whose last fine node has one parent
@pytest.mark.parametrize("nel", [(64, 32, 32), (65, 33, 32)])
@pytest.mark.parametrize("nvec", [7, 8])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_vcycle_of_many_vectors_equals_single(tofe, nel, nvec, prec):
    """One V-cycle on nvec vectors equals the V-cycle on each of them, bit for bit."""
    print(f"case restriction {nel} x {nvec} {prec}", flush=True)
    pb = configs.cantilever(nel, seed=3, lo=0.05, hi=1.0, rmin=1.5, penal=3.0, mg_levels=4)
    ctx = tofe.Context(nel, rmin=1.5, penal=3.0, mg_levels=4, fixed_dof=pb.fixed_dof)
    ctx.set_precision(tofe.PREC_MIXED if prec == "mixed" else tofe.PREC_FP64)
    ctx.set_design(pb.x)
    ctx.assemble()
    R = np.random.default_rng(5).standard_normal((nvec, ctx.ndof))
    R[:, pb.fixed_dof.astype(bool)] = 0
    Z = ctx.pc_apply(R.ravel()).reshape(nvec, -1)
    for v in range(nvec):
        assert np.array_equal(Z[v], ctx.pc_apply(R[v].copy())), v
    ctx.close()


@pytest.mark.parametrize("levels", [1, 2, 3])
@pytest.mark.parametrize("nvec", [1, 3, 16])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_residual_reduction_with_the_restriction(tofe, levels, nvec, prec):
    """The solve's r.r goes with the next V-cycle's first restriction, or (one level, or a step that
    may be the last) by itself: a block solve equals the single solves bit for bit, and the last
    step's residual is the one of the returned solution (1e-7: rtol 1e-9 on a system of condition
    below 1e6 in FP64 arithmetic leaves the recurrence within 1e-10 of it)."""
    print(f"case reduction levels {levels} x {nvec} {prec}", flush=True)
    pb = configs.cantilever((16, 8, 8), seed=3, lo=0.3, hi=1.0, rmin=1.5, penal=3.0, mg_levels=levels)
    ctx = tofe.Context((16, 8, 8), rmin=1.5, penal=3.0, mg_levels=levels, fixed_dof=pb.fixed_dof)
    ctx.set_precision(tofe.PREC_MIXED if prec == "mixed" else tofe.PREC_FP64)
    ctx.set_design(pb.x)
    ctx.assemble()
    F = np.random.default_rng(5).standard_normal((nvec, ctx.ndof))
    F[:, pb.fixed_dof.astype(bool)] = 0
    U, _, reason = ctx.solve(F, rtol=1e-9, maxit=200)
    assert reason > 0
    U = np.asarray(U).reshape(nvec, -1)
    for v in range(nvec):
        one, _, _ = ctx.solve(F[v].copy(), rtol=1e-9, maxit=200)
        assert np.array_equal(U[v], np.asarray(one).ravel()), v
        res = F[v] - np.asarray(ctx.apply_K(U[v].copy())).ravel()
        assert np.linalg.norm(res) <= 1e-7 * np.linalg.norm(F[v])
    ctx.close()
