"""The consistent mass and the stress stiffness on the element march at the edges of its
15 x 15-column tiles and of its z-chunks, for one vector and for blocks across the 16-vector pass,
against the closed-form mass assembly (1e-14) and the oracle's Ks (1e-13)."""
import numpy as np
import pytest

from test_gpu_mass import consistent_mass_csr
from topopt3d_amd import configs

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("zlen", [None, "1:1", "5:5"])
@pytest.mark.parametrize("nel", [(14, 15, 4), (16, 29, 3), (31, 5, 9), (2, 2, 2)])
def test_mass_and_stress_at_tile_edges(oracle, tofe, nel, zlen, monkeypatch):
    print(f"case nel={nel} zlen={zlen}", flush=True)
    if zlen:
        monkeypatch.setenv("TOFE_FINE_WHT_Z", zlen)
    h = (1.0, 0.5, 1.25)
    pb = configs.cantilever(nel, seed=6, lo=0.05, hi=1.0)
    ctx = tofe.Context(nel, h=h, mg_levels=1 if nel == (2, 2, 2) else 2, fixed_dof=pb.fixed_dof)
    ctx.set_design(pb.x)
    rng = np.random.default_rng(9)
    U = rng.standard_normal(pb.ndof)
    U[pb.fixed_dof.astype(bool)] = 0
    X = rng.standard_normal((17, pb.ndof))
    ctx.set_mass_form(tofe.MASS_CONSISTENT)
    ctx.assemble_mass(2.5)
    M = consistent_mass_csr(nel, h, ctx.field(tofe.FIELD_RHO), 2.5, pb.fixed_dof, None)[0]
    ctx.set_stress(U)
    Ks = oracle.assemble_Ks(*nel, U, ctx.field(tofe.FIELD_ES), pb.fixed_dof, h=h).to_scipy()
    for A, apply, tol in ((M, ctx.apply_M, 1e-14), (Ks, ctx.apply_Ks, 1e-13)):
        Y = apply(X)
        for j in range(17):
            assert rel(Y[j], A @ X[j]) <= tol
        assert np.array_equal(Y[16], apply(X[16]))
    ctx.close()
