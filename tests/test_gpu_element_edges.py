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


def assembled(prob, orc):
    import torch

    from svfsi_amd.step import NewtonStep

    st = NewtonStep(prob)
    # the element loop accumulates into what is there
    V0 = torch.rand_like(st.Val)
    R0 = torch.rand_like(st.R)
    st.Val.copy_(V0)
    st.R.copy_(R0)
    st.dmesh.assemble(prob.phys, prob.eq, st.Ag, st.Yg, st.Dg, st.Val, st.R, prop_el=st.prop, quad=prob.quad)
    Vo, Ro = orc.assemble(prob, st.rowPtr - 1, st.colPtr - 1)
    return [(a.cpu().numpy() - b.cpu().numpy(), c) for a, b, c in ((st.Val, V0, Vo), (st.R, R0, Ro))]


VISC = {"const": {}, "cy": dict(viscType=697, mu=0.035, mu_o=0.56, lam=3.313, visc_a=2.0, visc_n=0.3568),
        "cass": dict(viscType=696, mu=0.2, mu_o=0.3, lam=0.5)}


@pytest.mark.gpu
@pytest.mark.parametrize("model", list(VISC))
@pytest.mark.parametrize("nEl,tDof,uniform", [(1, 4, True), (13, 7, False), (65, 4, False), (130, 5, True)])
def test_fluid_assembly_sizes(gpu, orc, nEl, tDof, uniform, model):
    prob = fluid_case(nEl, tDof, uniform)
    prob.eq = dict(prob.eq, fb=(0.3, -0.2, 0.1), **VISC[model])
    for got, want in assembled(prob, orc):
        assert np.abs(got - want.reshape(got.shape)).max() <= 1e-12 * max(1.0, np.abs(want).max())


@pytest.mark.gpu
@pytest.mark.parametrize("kind,size", [("lelas", 1), ("lelas", 5), ("fluid", 0.45), ("fluid", 0.2)])
def test_face_terms_sizes(gpu, orc, kind, size):
    """Two faces, a handful to several hundred faces, nodes of up to eight faces, one launch each."""
    prob = problems.lelas_cube(size) if kind == "lelas" else problems.fluid_cylinder(h=size)
    import torch

    from svfsi_amd.step import NewtonStep

    st = NewtonStep(prob)
    rng = np.random.default_rng(1)
    st.Yg.copy_(torch.from_numpy(rng.normal(size=prob.Yg.shape)))
    prob.Yg = st.Yg.cpu().numpy()
    st.assemble()
    got = st.Val.cpu().numpy(), st.R.cpu().numpy()
    want = orc.assemble(prob, st.rowPtr - 1, st.colPtr - 1)
    for a, b in zip(got, want):
        assert np.abs(a - b.reshape(a.shape)).max() <= 1e-12 * np.abs(b).max()


@pytest.mark.gpu
@pytest.mark.parametrize("nEl,shift", [(1, 0), (13, 1), (130, 1), (1200, 0)])
def test_zero_sizes(gpu, nEl, shift):
    """Val and R cleared to their ends and no further, on 16- and 8-byte boundaries."""
    import torch

    from svfsi_amd import fsils
    from svfsi_amd.assembly import DeviceMesh

    prob = fluid_case(nEl, 4, True)
    rowPtr, colPtr = fsils.lhsa(prob.nNo, prob.mesh.ien)
    lhs = fsils.fsils_lhs_create(prob.nNo, len(colPtr), rowPtr, colPtr)
    dm = DeviceMesh(lhs, prob.mesh)
    for dof in (3, 4):
        nV, nR = len(colPtr) * dof * dof, prob.nNo * dof
        V, R = (torch.ones(n + 4, dtype=torch.float64, device=gpu) for n in (nV, nR))
        dm.zero(dof, V[shift:shift + nV], R[shift:shift + nR])
        for t, n in ((V, nV), (R, nR)):
            assert t[shift:shift + n].abs().max().item() == 0.0
            assert t[:shift].eq(1).all() and t[shift + n:].eq(1).all()


def lelas_case(nEl, tDof, uniform, seed=4):
    prob = problems.lelas_cube(4)
    rng = np.random.default_rng(seed)
    prob.mesh.x = prob.mesh.x + rng.uniform(-0.03, 0.03, prob.mesh.x.shape)
    prob.Ag, prob.Dg = (wide(rng.normal(size=(prob.nNo, 3)), tDof, rng) for _ in range(2))
    prob.Yg = np.zeros_like(prob.Dg)
    prob.prop_el = None if uniform else 1e3 * np.exp(0.3 * rng.normal(size=prob.mesh.nEl))
    prob.eq = dict(prob.eq, E=1e3, fb=(0.3, -0.2, 0.1))
    return first_elements(prob, nEl)


@pytest.mark.gpu
@pytest.mark.parametrize("nEl,tDof,uniform", [(1, 3, True), (13, 7, False), (65, 3, False), (130, 4, True)])
def test_lelas_assembly_sizes(gpu, orc, nEl, tDof, uniform):
    for got, want in assembled(lelas_case(nEl, tDof, uniform), orc):
        assert np.abs(got - want.reshape(got.shape)).max() <= 1e-12 * np.abs(want).max()


@pytest.mark.gpu
@pytest.mark.parametrize("points", [60, 200, 400])
@pytest.mark.parametrize("kind", ["lelas", "fluid"])
def test_assembly_hub_node(gpu, orc, kind, points):
    """Tets that all share one node: its diagonal block sums fewer, more, and
    several times more contributions than a gather tile holds (128)."""
    from scipy.spatial import ConvexHull

    rng = np.random.default_rng(points)
    s = rng.normal(size=(points, 3))
    s /= np.linalg.norm(s, axis=1, keepdims=True)
    tri = ConvexHull(s).simplices
    x = np.concatenate([s, np.zeros((1, 3))])
    ien = np.concatenate([tri, np.full((len(tri), 1), points)], axis=1)
    m = meshmod.TetMesh(x=x, ien=meshmod._orient(x, ien.astype(np.int32)).astype(np.int32))
    prob = fluid_case(1, 4, True) if kind == "fluid" else lelas_case(1, 3, True)
    prob.mesh = m
    for k in ("Ag", "Yg", "Dg"):
        setattr(prob, k, rng.normal(size=(m.nNo, prob.dof)))
    for got, want in assembled(prob, orc):
        assert np.abs(got - want.reshape(got.shape)).max() <= 1e-12 * max(1.0, np.abs(want).max())


VOL = {"quad": dict(volType=1), "st91": dict(volType=2), "m94": dict(volType=3), "none": dict(Kpen=0.0)}


@pytest.mark.gpu
@pytest.mark.parametrize("vol", list(VOL))
@pytest.mark.parametrize("nEl,tDof,quad", [(1, 3, 0), (5, 3, 0), (6, 4, 0), (162, 3, 0), (9, 3, 1), (10, 7, 1),
                                           (11, 3, 1), (162, 4, 1)])
def test_struct_assembly_sizes(gpu, orc, nEl, tDof, quad, vol):
    prob = problems.struct_cube(n=3, quad=quad)
    rng = np.random.default_rng(7)
    prob.Ag = rng.normal(size=(prob.nNo, 3))
    # |grad u| <= 0.004 * sum_a |grad N_a| <= 0.004 * (6 + 12) * 3 sqrt(2) < 1/3
    # per entry: F is diagonally dominant, no element is inverted
    prob.Dg = rng.uniform(-0.004, 0.004, size=(prob.nNo, 3))
    prob.Ag, prob.Dg = wide(prob.Ag, tDof, rng), wide(prob.Dg, tDof, rng)
    prob.Yg = np.zeros_like(prob.Dg)
    prob.eq = dict(prob.eq, fb=(0.3, -0.2, 0.1), **VOL[vol])
    for got, want in assembled(first_elements(prob, nEl), orc):
        assert np.abs(got - want.reshape(got.shape)).max() <= 1e-12 * np.abs(want).max()


@pytest.mark.gpu
@pytest.mark.parametrize("quad", [0, 1])
def test_struct_without_scratch(gpu, orc, monkeypatch, quad):
    """162 elements of 7.4 or 8.4 KB do not fit 1 MB: the coloured kernels run,
    to the bits of the call that asks for them."""
    prob = first_elements(problems.struct_cube(n=3, quad=quad), 162)
    rng = np.random.default_rng(11)
    prob.Dg = rng.uniform(-0.004, 0.004, size=(prob.nNo, 3))

    def run():  # on the same random Val and R each time
        import torch

        torch.manual_seed(11)
        return assembled(prob, orc)

    monkeypatch.setenv("SVFSI_ASM_SCRATCH_MB", "1")
    capped = run()
    monkeypatch.setenv("SVFSI_ASM_SCRATCH_MB", "2")
    monkeypatch.setenv("SVFSI_ASM_GATHER", "0")
    coloured = run()
    monkeypatch.delenv("SVFSI_ASM_GATHER")
    roomy = run()
    for (got, want), (col, _), (out, _) in zip(capped, coloured, roomy):
        assert np.abs(got - want.reshape(got.shape)).max() <= 1e-12 * np.abs(want).max()
        assert np.array_equal(got, col)
        assert np.abs(out - got).max() <= 1e-12 * np.abs(want).max()
    assert not np.array_equal(capped[0][0], roomy[0][0])  # the two paths round differently
