"""Nodes that join many elements: 6×6 blocks of many elements, and sums of more than 32 contributions, a
wave each, in the order of the elements. Lλx is bitwise the segmented scatter's, Lλ bitwise the
sum in that order of the elements' residuals (:iter), and both agree with the oracle to 1e-12. Sizes on both sides
of a lane's four, 32, a wave's 64 and several gathers, dofs with many
loads, and Newton iterations that write such a sum into the chain solve's right-hand side."""
import numpy as np
import pytest

from tests.helpers import oracle_model, relerr
from tests.test_gpu_scatter_dispatch import bits, info, same_as_segmented

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mc():
    import muscade_amd
    return muscade_amd


def hub(mc, kind, n):
    from muscade_amd.workloads import base_section
    rng = np.random.default_rng(n)
    m = mc.Model(kind)
    v = rng.normal(size=(n, 3))
    v *= 10. / np.linalg.norm(v, axis=1)[:, None]
    pairs = np.stack([np.ones(n, int), np.arange(2, n + 2)], axis=1)
    if kind in ("parallel", "anchored"):   # n beams between the same two nodes; a chain goes on, its anchor held
        k = 1 if kind == "parallel" else 12
        mc.addnode(m, np.stack([np.arange(k + 1.), np.zeros(k + 1), np.zeros(k + 1)], axis=1))
        pairs = np.concatenate([np.tile([[1, 2]], (n, 1))] + [np.array([[i, i + 1]]) for i in range(2, k + 1)])
        mc.addelement(m, mc.EulerBeam3D, pairs, mat=base_section(), orient2=np.array([0., 1., 0.]))
    else:
        mc.addnode(m, np.zeros((1, 3)))
        mc.addnode(m, v)
        if kind == "bars":
            mc.addelement(m, mc.Bar3D, pairs, mat=mc.AxisymmetricBarCrossSection(EA=1e6, mu=5., w=10.))
        else:
            mc.addelement(m, mc.EulerBeam3D, pairs, mat=base_section(), orient2=rng.normal(size=(n, 3)))
    if kind == "loads":             # and n loads on one dof of a spoke
        for k in range(n):
            mc.addelement(m, mc.DofLoad, [2], field="t3", value=lambda t, k=k: 0.1 * k * t)
    if kind != "parallel":
        mc.addelement(m, mc.Hold, [1 if kind == "anchored" else 2], field="t1")
    st = mc.initialize(m, nXder=3, time=0.5)
    for d in range(3):
        st.X[d][:] = rng.normal(0., 1e-2, st.X[d].size)
    return m, st


CASES = [("star", n) for n in (3, 4, 5, 6, 7, 8, 9, 12, 32, 33, 63, 64, 65, 127, 128, 129, 700)] + \
        [("parallel", n) for n in (4, 11, 32, 33, 300)] + [("anchored", n) for n in (9, 31, 32, 33, 70)] + \
        [("bars", n) for n in (32, 33, 130)] + [("loads", 31), ("loads", 32), ("loads", 66)]


@pytest.mark.parametrize("OX", [0, 1, 2])
@pytest.mark.parametrize("kind,n", CASES)
def test_long_sums(mc, kind, n, OX):
    print("case", kind, n, OX, flush=True)
    model, st = hub(mc, kind, n)
    i = same_as_segmented(mc, model, st, OX)
    more, one = int(n > 32), int(n + 1 > 32)    # a held or loaded dof has one contribution more
    rlong = {"star": 6 * more, "loads": 6 * more + one, "bars": 3 * more, "parallel": 12 * more,
             "anchored": 5 * more + one + 6 * one}[kind]
    by_nodes = kind != "bars" and OX > 0
    long = {"loads": one, "anchored": 71 * more + one}.get(kind, 0) * by_nodes
    assert (i["nodes"], i["rlong"], i["long"]) == (by_nodes, rlong, long), i
    out = mc.AssemblySweepX(OX, model, st.dis)
    out.c = mc.Newmarkβcoefficients(OX, 0.05)
    for mission in ("iter", "step"):
        Lλ, nz = out.assemble(st, mission)
        om = oracle_model(model, st.dis, t=st.time)
        r, rhs, onz, err = om.assemble(OX, 0 if mission == "step" else 1, out.c.array(), st.X[:OX + 1], None, None)
        assert r == 0, err
        assert relerr(Lλ, rhs) <= 1e-12 and relerr(nz, onz) <= 1e-12, mission
        if mission == "iter":
            s = np.zeros(out.nX)
            for it, d in enumerate(st.dis.dis):
                np.add.at(s, (d.X - 1).ravel(), out.element_blocks(it)[0].ravel())
            assert np.array_equal(bits(Lλ), bits(s))


@pytest.mark.parametrize("nload", [32, 33, 70])
def test_newton_iterations_with_a_long_sum(mc, nload):
    """A chain whose top carries many loads, in whole Newton iterations."""
    from muscade_amd.chainsolve import ChainSolver
    from muscade_amd.workloads import catenary_chains
    model, st = catenary_chains(nchain=1, nmin=40, nmax=40, seed=2)
    model.locked = False
    for k in range(nload - 2):      # beside the last beam and the top load
        mc.addelement(model, mc.DofLoad, [41], field="t1", value=lambda t, k=k: 0.1 * k * t)
    st2 = mc.initialize(model, nXder=3, time=1.)
    for d in range(3):
        st2.X[d][:st.X[d].size] = st.X[d]
    c = mc.Newmarkβcoefficients(2, 0.05)
    ends = []
    for graph in (False, True):
        out = mc.AssemblySweepX(2, model, st2.dis, graph=graph)
        out.c = c
        assert info(mc, out)["rlong"] == (nload > 32)
        cs = ChainSolver(out)
        out.set_state(st2, st2.time)
        for k in range(3):
            if graph:
                cs.iteration_graph(2, k == 0, c.array())
            else:
                out.assemble(st2, "step" if k == 0 else "iter", fetch=False, upload=False)
                cs.solve()
                cs.newton_update(2, k == 0, c.array())
        end = st2.copy()
        cs.fetch_X(end, 2)
        ends.append(end)
    for d in range(3):
        assert np.array_equal(bits(ends[0].X[d]), bits(ends[1].X[d]))
