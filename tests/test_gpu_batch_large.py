"""Merged batches whose launches fill the GPU: chunk lengths, stencil forms and restriction forms then
follow the launch's total, which a single solve of the instance does not have, and the results must
still be the single solves' bits."""
import pytest

from topopt3d_amd import configs

pytestmark = pytest.mark.gpu


# level-1 grids of 30,625, 18,081 and 637 nodes: with 1, 4 (vectors in fours) and 5 (one by one) load
# cases on either side of every rule's bound
@pytest.mark.parametrize("nrhs", [1, 4, 5])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("split", [None, "0", "1000000"])
def test_merged_batch_of_large_instances(tofe, monkeypatch, nrhs, precision, split):
    import torch

    print(f"case large batch loads={nrhs} precision={precision} split={split}", flush=True)
    monkeypatch.setenv("TOFE_BATCH_GRAPH", "merged")
    if split is not None:
        monkeypatch.setenv("TOFE_STENCIL_SPLIT_NODES", split)
    ctxs, F = [], []
    gen = torch.Generator().manual_seed(3)
    for i, nel in enumerate([(96, 48, 48), (80, 40, 40), (24, 12, 12), (96, 48, 48)]):
        pb = configs.cantilever(nel, seed=5 + i, lo=0.05, hi=1.0)
        c = tofe.Context(nel, fixed_dof=pb.fixed_dof, precision=precision)
        c.set_design(pb.x)
        c.assemble()
        f = torch.randn((nrhs, pb.ndof), dtype=torch.float64, generator=gen)
        f[:, torch.from_numpy(pb.fixed_dof.astype(bool))] = 0
        ctxs.append(c)
        F.append(f.cuda())
    batch = tofe.Batch(ctxs)
    Ub = [torch.zeros_like(f) for f in F]
    its, rs = batch.solve_dev([f.data_ptr() for f in F], [u.data_ptr() for u in Ub], nrhs,
                              rtol=1e-8, maxit=200, chunk=2)
    assert (rs == tofe.CONVERGED_RTOL).all()
    for c, f, u in zip(ctxs, F, Ub):
        Ue = torch.zeros_like(f)
        _, reason = c.solve_dev(f.data_ptr(), Ue.data_ptr(), nrhs=nrhs, rtol=1e-8, maxit=200)
        assert reason == tofe.CONVERGED_RTOL and torch.equal(u, Ue)
    batch.close()
    for c in ctxs:
        c.close()
