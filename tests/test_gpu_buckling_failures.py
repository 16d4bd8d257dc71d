"""Buckling sensitivities at their limits."""
import ctypes as C

import numpy as np
import pytest

from topopt3d_amd import _lib, configs, eigen

pytestmark = pytest.mark.gpu


def test_failed_adjoint_solve_is_reported(tofe):
    """One CG step does not reach 1e-12: the gradients stay unwritten, the caller learns of it by the
    reason or, without one, by the return code."""
    import torch

    print("case failed adjoint solve", flush=True)
    nel, nev = (9, 6, 5), 2
    pb = configs.column(nel, seed=3, lo=0.1, Emin=1e-9, rmin=1.5)
    ctx = tofe.Context(nel, rmin=1.5, Emin=1e-9, mg_levels=2, fixed_dof=pb.fixed_dof)
    ctx.set_design(pb.x)
    ctx.assemble()
    rng = np.random.default_rng(8)
    U = rng.standard_normal(ctx.ndof)
    phi = rng.standard_normal((nev, ctx.ndof))
    U[pb.fixed_dof.astype(bool)] = 0
    phi[:, pb.fixed_dof.astype(bool)] = 0
    ctx.set_stress(U)
    dU, dphi = torch.from_numpy(U).cuda(), torch.from_numpy(phi).cuda()
    g = torch.full((nev, ctx.nelem), -7.0, dtype=torch.float64, device="cuda")
    mu = np.array([0.5, 0.25])
    _, reason = ctx.buckling_sensitivity_dev(dU.data_ptr(), mu, dphi.data_ptr(), g.data_ptr(),
                                             rtol=1e-12, maxit=1)
    assert reason == tofe.DIVERGED_ITS and (g == -7.0).all()
    args = (ctx.h, C.c_void_p(dU.data_ptr()), mu.ctypes.data_as(C.POINTER(C.c_double)),
            C.c_void_p(dphi.data_ptr()), nev, 1e-12)
    L = _lib.lib()
    rc = L.tofe_buckling_sensitivity_dev(*args, 1, C.c_void_p(g.data_ptr()), None, None)
    assert rc == tofe.TOFE_ERR_NUMERIC and (g == -7.0).all()
    with pytest.raises(RuntimeError):
        eigen.buckling_sensitivities(ctx, dU, mu, dphi, rtol=1e-12, maxit=1)
    # with enough steps neither is needed
    rc = L.tofe_buckling_sensitivity_dev(*args, 2000, C.c_void_p(g.data_ptr()), None, None)
    assert rc == tofe.TOFE_OK and not (g == -7.0).any()
    ctx.close()


def test_more_vectors_than_a_grid_axis_holds(tofe):
    """70,001 vectors of a mesh of two elements: the adjoint right-hand sides of the first and the last
    ones are those of a call of their own, bit for bit."""
    print("case 70,001 vectors", flush=True)
    nel, nvec = (2, 1, 1), 70001
    fixed = np.zeros(36, np.uint8)
    fixed[[0, 1, 2, 9, 10, 11]] = 1
    ctx = tofe.Context(nel, rmin=1.0, mg_levels=1, fixed_dof=fixed)
    ctx.set_design(np.array([0.3, 0.8]))
    phi = np.random.default_rng(5).standard_normal((nvec, ctx.ndof))
    U = np.random.default_rng(6).standard_normal(ctx.ndof)
    ctx.set_stress(U)
    q, r = ctx.stability_terms(phi)
    for j in (0, 1, 65534, 65535, 65536, nvec - 1):
        qj, rj = ctx.stability_terms(phi[j])
        np.testing.assert_array_equal(r[j], rj[0])
        np.testing.assert_array_equal(q[j], qj[0])
        assert np.abs(rj).max() > 0
    ctx.close()
