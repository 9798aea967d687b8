"""The matrix-resident polynomial preconditioner (one launch per application)
against one launch per factor: the same polynomial with the products of long
rows summed in another order, so the mixed solve makes the same outer steps
(one more or less where the residual passes near the tolerance) and reaches
the same solution to its own tolerance."""
import threading
import time

import numpy as np
import pytest

from svfsi_amd import fsils, problems
from svfsi_amd import mesh as meshmod


def hub(points):
    """Tets around one node: its block row holds points + 1 blocks."""
    from scipy.spatial import ConvexHull

    rng = np.random.default_rng(points)
    s = rng.normal(size=(points, 3))
    s /= np.linalg.norm(s, axis=1, keepdims=True)
    tri = ConvexHull(s).simplices
    x = np.concatenate([s, np.zeros((1, 3))])
    ien = np.concatenate([tri, np.full((len(tri), 1), points)], axis=1)
    prob = problems.lelas_cube(2)
    prob.mesh = meshmod.TetMesh(x=x, ien=meshmod._orient(x, ien.astype(np.int32)).astype(np.int32))
    for k in ("Ag", "Yg", "Dg"):
        setattr(prob, k, np.zeros((points + 1, 3)))
    prob.Dg = 1e-3 * rng.normal(size=(points + 1, 3))
    prob.dir_faces, prob.trac_faces = [(np.arange(4, dtype=np.int32), 3)], []
    return prob


CASES = {
    "lelas_1part": lambda: problems.lelas_cube(3),
    "lelas_parts": lambda: problems.lelas_cube(13),
    "lelas_all_cus": lambda: problems.lelas_cube(27),
    "fluid_few": lambda: problems.fluid_cylinder(h=0.5),
    "fluid_mid": lambda: problems.fluid_cylinder(h=0.22),
    "hub_16_lanes": lambda: hub(40),
    "hub_64_lanes": lambda: hub(150),
    "hub_no_fit": lambda: hub(400),
    "lelas_5_blocks": lambda: problems.lelas_cube(32),
    "fluid_5_blocks": lambda: problems.fluid_cylinder(h=0.095),
    "tet10": lambda: problems.struct_cube(3, Kpen=1e5),
}


# blocks a lane of the patterns that get other than three; 0: no partition
BLOCKS = {"hub_no_fit": 0, "lelas_5_blocks": 5, "fluid_5_blocks": 5}


def solve(prob, monkeypatch, persist, wait=None, mixed=True, blocks=None):
    """The second of two equal solves, after checking which kernels ran: those
    of a partition with `blocks` blocks a lane (None: as PERSIST says; 0: none),
    given up once if the wait is 0."""
    import torch

    from svfsi_amd.step import NewtonStep

    monkeypatch.setenv("SVFSI_PERSIST", persist)
    if wait is None:
        monkeypatch.delenv("SVFSI_PERSIST_WAIT", raising=False)
    else:
        monkeypatch.setenv("SVFSI_PERSIST_WAIT", wait)
    st = NewtonStep(prob)
    out = []
    for _ in range(2):  # the second solve reuses the partition and its exchange buffer
        ls = st.step(mixed=mixed)
        torch.cuda.synchronize()
        out.append((st.R.cpu().numpy().copy(), ls.RI.itr, ls.RI.suc))
    r = st.lhs.resident_stats()
    if blocks is not None:
        assert r["blocks"] == blocks and (r["parts"] > 0) == (blocks > 0)
    used = persist == "1" and r["parts"] > 0 and (mixed or r["blocks"] == 3) and prob.ls["mItr"] > 0
    assert (r["launches"] > 0) == used, r
    if not (used and wait == "0"):
        assert r["give_ups"] == 0
    elif prob.ls["LS_type"] == fsils.LS_TYPE_NS and not mixed:  # a Schur solve per outer step, every 17th tries
        assert 1 <= r["give_ups"] <= 3
    else:
        assert r["give_ups"] == 1
    assert np.array_equal(out[0][0], out[1][0])
    return out[0]


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_matches_one_launch_per_factor(gpu, monkeypatch, name):
    prob = CASES[name]()
    x, itr, suc = solve(prob, monkeypatch, "1", blocks=BLOCKS.get(name, 3))
    y, itr0, suc0 = solve(prob, monkeypatch, "0")
    assert suc == suc0 == 1 and abs(itr - itr0) <= 1
    # both solve to 1e-8 in the scaled residual
    assert np.linalg.norm(x - y) <= 1e-6 * np.linalg.norm(y)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["lelas_parts", "lelas_all_cus", "fluid_mid", "tet10", "lelas_5_blocks", "fluid_5_blocks"])
def test_gives_up_and_falls_back(gpu, monkeypatch, name):
    """A wait of no ticks: the kernel ends at the first word not yet there,
    some workgroups before others have started, and the solve runs again with
    one launch per factor, to the same bits."""
    prob = CASES[name]()
    x, itr, suc = solve(prob, monkeypatch, "1", wait="0", blocks=BLOCKS.get(name, 3))
    y, itr0, suc0 = solve(prob, monkeypatch, "0")
    assert suc == suc0 == 1 and itr == itr0
    assert np.array_equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("mixed", [True, False])
def test_first_solve_on_recycled_memory(gpu, monkeypatch, mixed):
    """Patterns of one size made and freed in turn, each solved at once on a
    stream that does not wait for the null stream: a buffer that still held
    the freed pattern's words, with the tags the new one starts with, would
    be read as its neighbours' values."""
    import torch

    from svfsi_amd.step import NewtonStep

    monkeypatch.setenv("SVFSI_PERSIST", "1")
    monkeypatch.delenv("SVFSI_PERSIST_WAIT", raising=False)
    first = {}
    with torch.cuda.stream(torch.cuda.Stream()):
        for k in range(8):
            prob = problems.lelas_cube(13)
            prob.prop_el = 1e6 * (1.0 + 0.5 * (k % 2)) * np.ones(prob.mesh.nEl)
            st = NewtonStep(prob)
            st.step(mixed=mixed)
            torch.cuda.current_stream().synchronize()
            x = st.R.cpu().numpy()
            assert np.array_equal(x, first.setdefault(k % 2, x))
            st.lhs.free()


@pytest.mark.gpu
def test_two_threads(gpu, monkeypatch):
    """Two mixed solves at once on streams of their own: their matrix-resident
    launches take turns, and both solve as they do alone."""
    import torch

    from svfsi_amd.step import NewtonStep

    monkeypatch.setenv("SVFSI_PERSIST", "1")
    probs = [problems.lelas_cube(11), problems.fluid_cylinder(h=0.3)]
    want = [solve(p, monkeypatch, "0") for p in probs]
    monkeypatch.setenv("SVFSI_PERSIST", "1")
    steps = [NewtonStep(p) for p in probs]
    torch.cuda.synchronize()
    got = [None, None]

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(4):
                ls = steps[i].step(mixed=True)
            s.synchronize()
            got[i] = (steps[i].R.cpu().numpy(), ls.RI.itr, ls.RI.suc)

    ts = [threading.Thread(target=work, args=(i,)) for i in (0, 1)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for (x, itr, suc), (y, itr0, _) in zip(got, want):
        assert suc == 1 and abs(itr - itr0) <= 1
        assert np.linalg.norm(x - y) <= 1e-6 * np.linalg.norm(y)
    for st in steps:
        r = st.lhs.resident_stats()
        assert r["launches"] > 0 and r["give_ups"] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("name,persist", [("hub_no_fit", "1"), ("lelas_1part", "0"), ("lelas_1part", "1")])
def test_does_not_wait_for_another_solve(gpu, monkeypatch, name, persist):
    """A solve without a partition, with the path off, or matrix-resident
    itself, beside a matrix-resident one of half a million iterations (2 s or
    more): it ends while that one runs."""
    import torch

    from svfsi_amd.step import NewtonStep

    monkeypatch.setenv("SVFSI_PERSIST", "1")
    monkeypatch.delenv("SVFSI_PERSIST_WAIT", raising=False)
    cg = dict(LS_type=fsils.LS_TYPE_CG, absTol=1e-300)
    slow = NewtonStep(with_ls(CASES["lelas_parts"](), relTol=1e-300, mItr=100, **cg))
    fast = NewtonStep(with_ls(CASES[name](), relTol=1e-8, mItr=2000, **cg))
    slow.step(), fast.step()  # workspaces
    slow.assemble(), fast.assemble()
    torch.cuda.synchronize()
    slow.prob.ls["mItr"] = 500000
    began = threading.Event()

    def work():
        with torch.cuda.stream(torch.cuda.Stream()):
            began.set()
            slow.solve()

    t = threading.Thread(target=work)
    t.start()
    began.wait()
    time.sleep(0.1)
    monkeypatch.setenv("SVFSI_PERSIST", persist)
    with torch.cuda.stream(torch.cuda.Stream()):
        ls = fast.solve()
        running = t.is_alive()
    t.join()
    assert ls.RI.suc == 1 and running
    r, q = fast.lhs.resident_stats(), slow.lhs.resident_stats()
    assert (r["launches"] > 0) == (name == "lelas_1part") and r["give_ups"] == q["give_ups"] == 0
    assert q["launches"] >= 500000 // 256


@pytest.mark.gpu
@pytest.mark.parametrize("mixed", [True, False])
def test_tries_again_after_giving_up(gpu, monkeypatch, mixed):
    """16 solves without the matrix-resident kernels after a give-up, 64 after
    the next in a row; a solve that ends with them starts over at 16."""
    import torch

    from svfsi_amd.step import NewtonStep

    monkeypatch.setenv("SVFSI_PERSIST", "1")
    monkeypatch.delenv("SVFSI_PERSIST_WAIT", raising=False)
    st = NewtonStep(problems.lelas_cube(6))

    def step(wait=None):
        if wait is None:
            monkeypatch.delenv("SVFSI_PERSIST_WAIT", raising=False)
        else:
            monkeypatch.setenv("SVFSI_PERSIST_WAIT", wait)
        before = st.lhs.resident_stats()
        ls = st.step(mixed=mixed)
        torch.cuda.synchronize()
        assert ls.RI.suc == 1
        r = st.lhs.resident_stats()
        return r["launches"] > before["launches"], r["give_ups"], st.R.cpu().numpy()

    used, give_ups, resident = step()
    assert used and give_ups == 0
    for rest, give_ups_ in ((16, 1), (64, 2)):
        used, give_ups, other = step(wait="0")
        assert used and give_ups == give_ups_
        for _ in range(rest):
            used, give_ups, x = step()
            assert not used and give_ups == give_ups_ and np.array_equal(x, other)
    used, give_ups, x = step()
    assert used and give_ups == 2 and np.array_equal(x, resident)
    assert step(wait="0")[:2] == (True, 3)
    assert [step()[0] for _ in range(17)] == [False] * 16 + [True]


def with_ls(prob, **ls):
    prob.ls = dict(prob.ls, **ls)
    return prob


FP64 = {
    **{k: lambda k=k: with_ls(CASES[k](), LS_type=fsils.LS_TYPE_CG, relTol=1e-8, mItr=2000)
       for k in ("lelas_1part", "lelas_parts", "lelas_all_cus", "hub_16_lanes", "hub_64_lanes", "hub_no_fit", "tet10")},
    # the Schur complement is iterated to the NS solver's inner tolerances
    **{f"ns_{k}": lambda k=k: with_ls(CASES[k](), LS_type=fsils.LS_TYPE_NS, relTol=1e-5, absTol=1e-30, mItr=20)
       for k in ("fluid_few", "fluid_mid")},
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(FP64))
def test_fp64_matches_one_launch_per_step(gpu, monkeypatch, name):
    """CG and the Schur complement's CG: sums over the parts in another order,
    so the same solution to the solver's tolerance."""
    prob = FP64[name]()
    x, itr, suc = solve(prob, monkeypatch, "1", mixed=False, blocks=BLOCKS.get(name, 3))
    y, itr0, suc0 = solve(prob, monkeypatch, "0", mixed=False)
    assert suc == suc0 == 1 and abs(itr - itr0) <= 2
    tol = 1e-4 if name.startswith("ns_") else 1e-6  # relTol 1e-5 and 1e-8, times the conditioning
    assert np.linalg.norm(x - y) <= tol * np.linalg.norm(y)


@pytest.mark.gpu
@pytest.mark.parametrize("mItr", [0, 1, 7, 256, 257, 600])
def test_cg_iteration_limit(gpu, monkeypatch, mItr):
    """The limit inside a launch, at its end, and beyond; X after mItr steps
    agrees while the iteration has not lost its digits."""
    prob = with_ls(CASES["lelas_parts"](), LS_type=fsils.LS_TYPE_CG, relTol=1e-300, absTol=1e-300, mItr=mItr)
    x, itr, suc = solve(prob, monkeypatch, "1", mixed=False)
    y, itr0, suc0 = solve(prob, monkeypatch, "0", mixed=False)
    assert (itr, suc) == (itr0, suc0) == (mItr, 0)
    assert np.linalg.norm(x - y) <= 1e-6 * np.linalg.norm(y)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["lelas_parts", "lelas_all_cus", "ns_fluid_few", "ns_fluid_mid"])
def test_fp64_gives_up_and_falls_back(gpu, monkeypatch, name):
    prob = FP64[name]()
    x, itr, suc = solve(prob, monkeypatch, "1", wait="0", mixed=False, blocks=3)
    y, itr0, suc0 = solve(prob, monkeypatch, "0", mixed=False)
    assert (itr, suc) == (itr0, suc0)
    assert np.array_equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("h", [0.3, 0.22, 0.11])
def test_ns_difference_is_rounding(gpu, monkeypatch, h):
    """At the NS solver's default tolerances (it stops at a relative residual of
    0.4) the solution keeps what 100 to 280 iterations of CG make of rounding:
    1e-14 on a coarse mesh, 1e-3 at 26,667 nodes.  The matrix-resident Schur CG
    moves it as one ulp in the state does: with the same counts, and by no more
    than eight times the largest of four such perturbations (a sample of a
    scatter that spans a factor of ten)."""
    import torch

    from svfsi_amd.step import NewtonStep

    rng = np.random.default_rng(1)
    prob = problems.fluid_cylinder(h=h)
    free = prob.dir_mask()[:, :1] != 0
    prob.Yg[:, :3] = np.where(free, rng.uniform(-1.0, 1.0, (prob.nNo, 3)), prob.Yg[:, :3])
    prob.ls = dict(LS_type=fsils.LS_TYPE_NS, relTol=0.4, absTol=1e-10, mItr=10)
    st = NewtonStep(prob)

    def step(persist, Yg):
        monkeypatch.setenv("SVFSI_PERSIST", persist)
        st.Yg.copy_(torch.from_numpy(Yg))
        ls = st.step()
        torch.cuda.synchronize()
        assert ls.RI.suc == 1
        return st.R.cpu().numpy(), (ls.RI.itr, ls.GM.itr, ls.CG.itr)

    ulp = np.finfo(float).eps
    x, its = step("0", prob.Yg)
    y, its1 = step("1", prob.Yg)
    assert its1 == its and st.lhs.resident_stats()["launches"] > 0
    moved = [np.linalg.norm(step("0", prob.Yg * (1 + ulp * rng.integers(-1, 2, prob.Yg.shape)))[0] - x) for _ in range(4)]
    assert np.linalg.norm(y - x) <= 8 * max(moved)
    for persist, want in (("0", x), ("1", y)):  # each repeats itself
        assert np.array_equal(step(persist, prob.Yg)[0], want)
