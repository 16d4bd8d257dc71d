"""V-cycles on several vectors on either side of the rules that give such launches another stencil
form, and with the threshold between the forms given: every vector keeps its single launch's bits."""
import pytest

from topopt3d_amd import configs

pytestmark = pytest.mark.gpu


# level 1 holds 70,785 nodes, 277 blocks of nodes a vector: 8, 9 and 10 vectors stay below the bound of
# 3,000, 12 and 16 take the node form with three and four vectors per thread, 5 and 7 with one
@pytest.mark.parametrize("split", [None, "0", "1000000"])
@pytest.mark.parametrize("precision", [0, 1])
def test_block_vcycle_forms(tofe, monkeypatch, precision, split):
    import torch

    print(f"case block forms precision={precision} split={split}", flush=True)
    nel = (128, 64, 64)
    pb = configs.cantilever(nel, seed=5, lo=0.05, hi=1.0)
    if split is not None:
        monkeypatch.setenv("TOFE_STENCIL_SPLIT_NODES", split)
    c = tofe.Context(nel, fixed_dof=pb.fixed_dof, precision=precision)
    c.set_design(pb.x)
    c.assemble()
    R = torch.randn((16, pb.ndof), dtype=torch.float64, generator=torch.Generator().manual_seed(2)).cuda()
    R[:, torch.from_numpy(pb.fixed_dof.astype(bool)).cuda()] = 0
    Z1, Z = torch.empty_like(R), torch.empty_like(R)
    for j in range(16):
        c.pc_apply_dev(R[j].data_ptr(), Z1[j].data_ptr(), 1)
    assert torch.isfinite(Z1).all() and Z1.abs().max() > 0
    for nv in (5, 7, 8, 9, 10, 12, 16):
        Z.zero_()
        c.pc_apply_dev(R.data_ptr(), Z.data_ptr(), nv)
        assert torch.equal(Z[:nv], Z1[:nv]), nv
    c.close()


# 9,537 nodes on level 1: five vectors stay below the 50,000 nodes x vectors from which the FP32
# restriction takes a thread per node, six reach them; FP64 keeps a thread per DOF
@pytest.mark.parametrize("nel", [(64, 32, 32), (65, 33, 32)])
@pytest.mark.parametrize("nvec", [5, 6])
@pytest.mark.parametrize("precision", [0, 1])
def test_restriction_forms(tofe, nel, nvec, precision):
    import torch

    print(f"case restriction {nel} x {nvec} precision={precision}", flush=True)
    pb = configs.cantilever(nel, seed=3, lo=0.05, hi=1.0, mg_levels=4)
    c = tofe.Context(nel, mg_levels=4, fixed_dof=pb.fixed_dof, precision=precision)
    c.set_design(pb.x)
    c.assemble()
    R = torch.randn((nvec, pb.ndof), dtype=torch.float64, generator=torch.Generator().manual_seed(4)).cuda()
    R[:, torch.from_numpy(pb.fixed_dof.astype(bool)).cuda()] = 0
    Z, Z1 = torch.empty_like(R), torch.empty_like(R)
    c.pc_apply_dev(R.data_ptr(), Z.data_ptr(), nvec)
    for j in range(nvec):
        c.pc_apply_dev(R[j].data_ptr(), Z1[j].data_ptr(), 1)
    assert Z.abs().max() > 0 and torch.equal(Z, Z1)
    c.close()
