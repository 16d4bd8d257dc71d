"""The fine operator's node-centric forms (TOFE_FINE_WHT=0): without the two-step launch of the
element-centric form, the CG residual update forms the V-cycle's first fine-level step and the
direction takes another buffer's place from the second step on, so the buffer that the last step
writes depends on the parity of the step counts.  The FP64 CG must get the new z wherever it ends."""
import numpy as np
import pytest

from topopt3d_amd import configs

pytestmark = pytest.mark.gpu

NEL, L = (16, 8, 8), 3


def _context(tofe, pb, nu1, nu2, precision=0):
    c = tofe.Context(NEL, rmin=pb.rmin, penal=pb.penal, mg_levels=L, nu_pre=nu1, nu_post=nu2,
                     fixed_dof=pb.fixed_dof, precision=precision)
    c.set_design(pb.x)
    c.assemble()
    return c


# step counts of both parities on either side of nu1 = 2, and none after the correction
@pytest.mark.parametrize("nu1,nu2", [(2, 2), (2, 1), (3, 2), (2, 3), (3, 3), (1, 2), (2, 0)])
@pytest.mark.parametrize("precision", [0, 1])
def test_node_form_solves_as_element_form(oracle, tofe, monkeypatch, nu1, nu2, precision):
    """Both forms apply the same preconditioner up to rounding, so a solve takes the same number
    of iterations to one, ends for the same reason and meets the residual; a stale z changes them by far
    more.  Several right-hand sides at once and a batch's iterations give the single solves' bits."""
    import torch

    print(f"case node form V({nu1},{nu2}) precision {precision}", flush=True)
    pb = configs.cantilever(NEL, seed=7, lo=0.05, hi=1.0, mg_levels=L)
    E = oracle.simp(oracle.filter_csr(*NEL, pb.rmin).matvec(pb.x), pb.penal, 1e-10)[0]
    K = oracle.assemble_K(*NEL, oracle.ke(), E, pb.fixed_dof)
    ref = _context(tofe, pb, nu1, nu2, precision)
    Ur, its_r, reason_r = ref.solve(pb.F, rtol=1e-10, maxit=200)
    ref.close()
    monkeypatch.setenv("TOFE_FINE_WHT", "0")
    c = _context(tofe, pb, nu1, nu2, precision)
    U, its, reason = c.solve(pb.F, rtol=1e-10, maxit=200)
    print(f"its {its} reason {reason}; element form its {its_r} reason {reason_r}", flush=True)
    assert reason == reason_r and abs(its - its_r) <= 1
    if reason == tofe.CONVERGED_RTOL:
        assert np.linalg.norm(pb.F - K.matvec(U)) <= 1.01e-10 * np.linalg.norm(pb.F)
    F2 = np.stack([pb.F, np.roll(pb.F, -6)])
    F2[:, pb.fixed_dof.astype(bool)] = 0
    U2, _, _ = c.solve(F2, rtol=1e-10, maxit=200)
    np.testing.assert_array_equal(U2[0], U)
    Fd = torch.from_numpy(F2).cuda()
    Ud = torch.zeros_like(Fd)
    b = tofe.Batch([c])
    b.solve_dev([Fd.data_ptr()], [Ud.data_ptr()], 2, rtol=1e-10, maxit=200, chunk=2)
    np.testing.assert_array_equal(Ud.cpu().numpy(), U2)
    b.close()
    c.close()
