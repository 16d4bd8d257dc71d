"""Buckling eigenvalue sensitivities on the device against the same terms put together on the host
from the context's element terms, adjoint solves and filter."""
import numpy as np
import pytest

from topopt3d_amd import _lib, configs, eigen

pytestmark = pytest.mark.gpu


# odd sizes; 1 mode, one more than a block of the adjoint solve, one more than a launch's eigenvalues
@pytest.mark.parametrize("nel,nev", [((9, 6, 5), 1), ((8, 4, 4), 17), ((7, 5, 4), 33)])
def test_device_gradients_equal_host_terms(tofe, nel, nev):
    """rtol 1e-13 of the largest entry: the sums of 24 products per element round apart by some
    24 eps, the adjoint solutions are the same solve's."""
    import torch
    print(f"case buckling gradients {nel} x {nev}", flush=True)
    pb = configs.column(nel, seed=3, lo=0.1, Emin=1e-9, rmin=1.5)
    ctx = tofe.Context(nel, rmin=1.5, Emin=1e-9, penal=3.0, mg_levels=2, fixed_dof=pb.fixed_dof)
    ctx.set_design(pb.x)
    ctx.assemble()
    rng = np.random.default_rng(8)
    U = rng.standard_normal(ctx.ndof)
    phi = rng.standard_normal((nev, ctx.ndof))
    U[pb.fixed_dof.astype(bool)] = 0
    phi[:, pb.fixed_dof.astype(bool)] = 0
    mu = rng.uniform(0.1, 1.0, nev)
    ctx.set_stress(U)
    dU = torch.from_numpy(U).cuda()
    dphi = torch.from_numpy(np.ascontiguousarray(phi.T)).cuda().T  # not contiguous
    g = eigen.buckling_sensitivities(ctx, dU, mu, dphi, rtol=1e-12)
    assert isinstance(g, np.ndarray) and g.shape == (nev, ctx.nelem) and g.dtype == np.float64

    pksp, rhs = ctx.stability_terms(phi)
    pkp, _ = ctx.element_quadratic(phi, mass=False)
    V, _, reason = ctx.solve(rhs, rtol=1e-12, maxit=2000)
    assert reason > 0
    vku = ctx.element_bilinear(V, U)
    dEdz, dEsdz = ctx.field(_lib.FIELD_DEDZ), ctx.field(_lib.FIELD_DESDZ)
    for j in range(nev):
        terms = [-dEsdz * pksp[j], -mu[j] * dEdz * pkp[j], dEdz * vku[j]]
        ref = ctx.chain_filter(None, sum(terms))[1]
        scale = ctx.chain_filter(None, sum(np.abs(t) for t in terms))[1].max()
        assert np.abs(g[j] - ref).max() <= 1e-13 * scale, j
    ctx.close()
