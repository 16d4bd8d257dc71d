"""The smoothed levels' eigenvalue estimates: levels below TOFE_STENCIL_SPLIT_NODES nodes share
their launches, the others have their own.  Levels of 45 to 1,377 nodes,
with all, some or none of them sharing, against the oracle's estimates of the same Jacobi-CG steps."""
import pytest

from test_gpu_parity import setup_pair

pytestmark = pytest.mark.gpu


# levels of (32,16,16): 1,377, 225 and 45 nodes and the coarsest; (9,6,5) has odd sizes; L=2 has no
# coarse level to smooth, L=1 no estimate at all
@pytest.mark.parametrize("nel,L", [((32, 16, 16), 5), ((9, 6, 5), 3), ((8, 4, 4), 2), ((4, 4, 4), 1)])
@pytest.mark.parametrize("threshold", ["0", "300", "1000000000"])
def test_estimates_shared_and_own_launches(oracle, tofe, monkeypatch, nel, L, threshold):
    """FP64: the dot products' partial sums are grouped differently from the oracle's (rel 1e-10, as
    in the other tests of these estimates); mixed: rounding of the FP32 operators (1e-4)."""
    print(f"case estimates {nel} levels {L} threshold {threshold}", flush=True)
    monkeypatch.setenv("TOFE_STENCIL_SPLIT_NODES", threshold)
    pb, ctx, Pf, rho, E, dEdz, Es, dEsdz, K = setup_pair(oracle, tofe, nel, L)
    mg = oracle.MG(K, tuple(n + 1 for n in nel), L)
    for prec, tol in ((tofe.PREC_FP64, 1e-10), (tofe.PREC_MIXED, 1e-4), (tofe.PREC_FP64, 1e-10)):
        ctx.set_precision(prec)
        ctx.assemble()
        for lvl in range(L - 1):
            assert ctx.level_lambda(lvl) == pytest.approx(mg.lam(lvl), rel=tol)
    ctx.close()
