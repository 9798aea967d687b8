"""GMRESV's step end in one launch (up to 160 chunks of 512 unknowns) and in
two, around the line between them: the same bits as each other, and against the
oracle, whose dot products are summed in another order, the solution to the
solver's tolerance and the step count to 2 %."""
import numpy as np
import pytest

from svfsi_amd import fsils, problems


# from two cells a side on: 24 unknowns exhaust the Krylov space before a cycle
# ends, and what follows is rounding
@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 7, 29, 30])  # 81, 1,536, 81,000 and 89,373 unknowns (159 and 175 chunks)
def test_gmres_step_end(gpu, orc, monkeypatch, n):
    import torch

    from svfsi_amd.step import NewtonStep

    prob = problems.lelas_cube(n)
    # a limit of a few steps on the large systems: the column of every step and
    # the cycle's end are compared, not the convergence
    prob.ls = dict(prob.ls, LS_type=fsils.LS_TYPE_GMRES, relTol=1e-8, mItr=2 if n > 7 else 50, sD=20)
    st = NewtonStep(prob)
    st.assemble()
    V, R = st.Val.cpu().numpy().copy(), st.R.cpu().numpy().copy()
    ends = []
    for one in "01":
        monkeypatch.setenv("SVFSI_GM_ONE_END", one)
        st.assemble()
        ls = st.solve()
        torch.cuda.synchronize()
        ends.append((st.R.cpu().numpy().copy(), ls.RI.itr, ls.RI.fNorm))
    assert np.array_equal(ends[0][0], ends[1][0]) and ends[0][1:] == ends[1][1:]
    x, _, so = orc.fsils_solve(st.rowPtr - 1, st.colPtr - 1, prob.dof, prob.dir_mask(), prob.ls, R, V)
    assert ls.RI.suc == so.suc and abs(ls.RI.itr - so.itr) <= max(1, 0.02 * so.itr)
    if n <= 7:  # converged, perhaps a step earlier or later
        assert ls.RI.suc == 1 and max(ls.RI.fNorm, so.fNorm) <= 1e-8 * so.iNorm
    else:
        assert abs(ls.RI.fNorm - so.fNorm) <= 1e-6 * so.fNorm
    # before convergence X is fixed by the Krylov space, to its conditioning
    assert np.linalg.norm(st.R.cpu().numpy() - x) <= 1e-6 * np.linalg.norm(x)
