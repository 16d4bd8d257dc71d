"""The LDS-tiled filter kernels at their edges: every halo width (neighbours 1 to 5 elements
away) and the first radius beyond them, on meshes one element below, at and above the 32 x 8 x 4
tile and smaller than the halo, with cubic and box elements -- bit for bit the oracle's filter,
maximum-length-scale filter, interpolation and chain rule (Filter.cpp:21-150,
Material_Interpolation.cpp:20-187)."""
import numpy as np
import pytest

from topopt3d_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nel", [(32, 8, 4), (33, 9, 5), (31, 7, 3), (5, 17, 9), (66, 3, 2)])
@pytest.mark.parametrize("rmin,rmax,h", [
    (1.5, 2.0, (1.0, 1.0, 1.0)), (2.5, 3.5, (1.0, 1.0, 1.0)), (3.5, 4.5, (1.0, 1.0, 1.0)),
    (4.5, 5.5, (1.0, 1.0, 1.0)), (5.5, 6.1, (1.0, 1.0, 1.0)),
    (6.1, 5.2, (1.0, 1.0, 1.0)), (2.1, 2.6, (1.25, 1.0, 0.6))])
def test_tiled_filters_bit_exact(oracle, tofe, nel, rmin, rmax, h):
    print(f"case nel={nel} rmin={rmin} rmax={rmax} h={h}", flush=True)
    ne = int(np.prod(nel))
    x = configs.uniform(9, ne, 0.05, 1.0)
    P = oracle.filter_csr(*nel, rmin, h=h)
    R, REdge = oracle.rfilter_csr(*nel, rmax, h=h)
    vd_min = 0.3 * np.diff(R.arrays()[0]).max()
    dV, dE = np.random.default_rng(3).standard_normal((2, ne))
    for vd in (-1.0, vd_min):
        ctx = tofe.Context(nel, h=h, rmin=rmin, mg_levels=2, rmax=rmax, vd_min=vd, vd_penal=2.0)
        ctx.set_design(x)
        o = oracle.matint(P, R if vd > 0 else None, REdge if vd > 0 else None, x, 3.0, 2.0, vd)
        for k, f in dict(rho=tofe.FIELD_RHO, y=tofe.FIELD_Y, rhoq=tofe.FIELD_RHOQ, E=tofe.FIELD_E,
                         dEdz=tofe.FIELD_DEDZ, Es=tofe.FIELD_ES, dEsdz=tofe.FIELD_DESDZ).items():
            assert np.array_equal(ctx.field(f), o[k]), (vd, k)
        assert np.array_equal(ctx.field(tofe.FIELD_X), x)
        gV, gE = ctx.chain_filter(dV, dE)
        oV, oE = oracle.chain_filter(P, R if vd > 0 else None, o["rho"], o["y"], o["rhoq"], dV, dE)
        assert np.array_equal(gV, oV) and np.array_equal(gE, oE)
        assert np.array_equal(ctx.filter(x), P.matvec(x))
        assert np.array_equal(ctx.filter_T(dE), P.rmatvec(dE))
        ctx.close()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_tiled_filter_keeps_non_finite_values_to_their_neighbours(oracle, tofe, bad):
    """An infinite or undefined density reaches its neighbours only, not the corners of the
    staged box."""
    nel = (20, 12, 10)
    P = oracle.filter_csr(*nel, 3.5)
    x = configs.uniform(9, int(np.prod(nel)), 0.05, 1.0)
    x[10 + 20 * (6 + 12 * 5)] = bad
    ctx = tofe.Context(nel, rmin=3.5, mg_levels=2)
    assert np.array_equal(ctx.filter(x), P.matvec(x), equal_nan=True)
    assert np.array_equal(ctx.filter_T(x), P.rmatvec(x), equal_nan=True)
    ctx.close()
