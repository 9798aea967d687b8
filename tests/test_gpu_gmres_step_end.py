"""GMRESV's step end in one launch (up to 160 chunks of 512 unknowns) and in
two, around the line between them, against the oracle: the dot products are summed
in another order there, so the solution agrees to the solver's tolerance and
the step count to 2 %."""
import numpy as np
import pytest

from svfsi_amd import fsils, problems


# from two cells a side on: 24 unknowns exhaust the Krylov space before a cycle
# ends, and what follows is rounding
@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 7, 29, 30])  # 81, 1,536, 81,000 and 89,373 unknowns (159 and 175 chunks)
def test_gmres_step_end(gpu, orc, n):
    import torch

    from svfsi_amd.step import NewtonStep

    prob = problems.lelas_cube(n)
    # a limit of a few steps on the large systems: the column of every step and
    # the cycle's end are compared, not the convergence
    prob.ls = dict(prob.ls, LS_type=fsils.LS_TYPE_GMRES, relTol=1e-8, mItr=2 if n > 7 else 50, sD=20)
    st = NewtonStep(prob)
    st.assemble()
    V, R = st.Val.cpu().numpy().copy(), st.R.cpu().numpy().copy()
    ls = st.solve()
    torch.cuda.synchronize()
    x, _, so = orc.fsils_solve(st.rowPtr - 1, st.colPtr - 1, prob.dof, prob.dir_mask(), prob.ls, R, V)
    assert ls.RI.suc == so.suc and abs(ls.RI.itr - so.itr) <= max(1, 0.02 * so.itr)
    assert abs(ls.RI.fNorm - so.fNorm) <= 1e-6 * max(so.fNorm, 1e-8 * so.iNorm) or n <= 7
    # before convergence X is fixed by the Krylov space, to its conditioning
    assert np.linalg.norm(st.R.cpu().numpy() - x) <= 1e-6 * np.linalg.norm(x)
