"""Element kernels at mesh sizes where their lane groups and workgroups end
unevenly, against the oracle: one element, part of a wavefront, one element
beyond a workgroup, several workgroups.  The tolerance is the 64-bit rounding
of sums of up to a hundred terms, 1e-12 of the largest entry."""
import numpy as np
import pytest

from svfsi_amd import mesh as meshmod
from svfsi_amd import problems


def first_elements(prob, nEl):
    """prob on the first nEl elements of its mesh (nodes renumbered)."""
    m = prob.mesh
    ien = m.ien[:nEl]
    nodes, inv = np.unique(ien, return_inverse=True)
    prob.mesh = meshmod.TetMesh(x=m.x[nodes], ien=inv.reshape(ien.shape).astype(np.int32))
    for k in ("Ag", "Yg", "Dg"):
        setattr(prob, k, getattr(prob, k)[nodes])
    prob.dir_faces, prob.trac_faces, prob.bflow_faces = [], [], []
    if prob.prop_el is not None:
        prob.prop_el = prob.prop_el[:nEl]
    return prob


def wide(a, tDof, rng):
    """a (nNo, dof) inside a state array of tDof columns, the rest filled."""
    w = rng.normal(size=(a.shape[0], tDof))
    w[:, : a.shape[1]] = a
    return w


def fluid_case(nEl, tDof, uniform, seed=2):
    prob = problems.fluid_cylinder(h=0.4)
    rng = np.random.default_rng(seed)
    prob.Ag[:, :3] = rng.normal(size=(prob.nNo, 3))
    prob.Yg[:, 3] = rng.normal(size=prob.nNo)
    prob.Ag, prob.Yg = wide(prob.Ag, tDof, rng), wide(prob.Yg, tDof, rng)
    prob.Dg = np.zeros_like(prob.Yg)
    prob.prop_el = None if uniform else 0.04 * np.exp(0.1 * rng.normal(size=prob.mesh.nEl))
    return first_elements(prob, nEl)


@pytest.mark.gpu
@pytest.mark.parametrize("nEl,tDof,uniform", [(1, 4, True), (13, 7, False), (65, 4, False), (130, 5, True)])
def test_fluid_dmu_sizes(gpu, orc, nEl, tDof, uniform):
    import torch

    from svfsi_amd.step import NewtonStep

    prob = fluid_case(nEl, tDof, uniform)
    st = NewtonStep(prob)
    rng = np.random.default_rng(3)
    lam, du = rng.normal(size=(2, prob.nNo, 4))
    dl, dd = (torch.from_numpy(a.copy()).to(gpu) for a in (lam, du))
    g = torch.full((nEl,), np.nan, dtype=torch.float64, device=gpu)
    st.dmesh.fluid_dmu_dot(prob.eq, st.Ag, st.Yg, st.prop, dl, dd, g)
    go = orc.fluid_dmu_dot(prob, lam, du)
    assert np.abs(g.cpu().numpy() - go).max() <= 1e-12 * np.abs(go).max()
