"""The autotuner measures the shapes that the context already runs, short chunks included."""
import numpy as np
import pytest

from topopt3d_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
def test_autotune_keeps_short_chunks(tofe, precision):
    """A mesh whose whole operator is a few blocks: one to three planes a chunk take two thirds of the
    time of four and more, so the tuner must end there, and the results stay what they were."""
    print(f"case autotune precision={precision}", flush=True)
    pb = configs.cantilever((24, 12, 12), seed=3, lo=0.05, hi=1.0, mg_levels=3)
    c = tofe.Context(pb.nel, mg_levels=3, fixed_dof=pb.fixed_dof, precision=precision)
    c.set_design(pb.x)
    c.assemble()
    X = np.random.default_rng(1).standard_normal((2, pb.ndof))
    X[:, pb.fixed_dof.astype(bool)] = 0
    KX, ZX = c.apply_K(X), c.pc_apply(X)
    U0, _, r0 = c.solve(pb.F, rtol=1e-10)
    zlen, split = c.autotune(nrep=20)
    assert 1 <= zlen <= 3 and split >= 0
    np.testing.assert_array_equal(c.apply_K(X), KX)
    ZX2 = c.pc_apply(X)
    assert np.abs(ZX2 - ZX).max() <= 1e-12 * np.abs(ZX).max()
    U1, _, r1 = c.solve(pb.F, rtol=1e-10)
    assert r1 == r0 and np.abs(U1 - U0).max() <= 1e-8 * np.abs(U0).max()
    assert 1 <= c.autotune(nrep=20)[0] <= 3
    c.close()


def test_autotune_leaves_a_poor_length(tofe, monkeypatch):
    """A given length of 24 planes, one block along z, is replaced on the same mesh."""
    print("case autotune from 24 planes", flush=True)
    monkeypatch.setenv("TOFE_FINE_WHT_Z", "24:24")
    pb = configs.cantilever((24, 12, 12), seed=3, lo=0.05, hi=1.0, mg_levels=3)
    c = tofe.Context(pb.nel, mg_levels=3, fixed_dof=pb.fixed_dof)
    c.set_design(pb.x)
    c.assemble()
    KX = c.apply_K(pb.F)
    assert 1 <= c.autotune(nrep=20)[0] <= 3
    np.testing.assert_array_equal(c.apply_K(pb.F), KX)
    c.close()
