"""Which way the assembly's sums are launched (mh_get_scatter), and that every way gives the same bits:
the nz by nodes against a shape of the segmented scatter, the rhs in the nz's launch (graphs of small
models) against its own, and whole Newton iterations, whose sums go into the chain solve's blocks,
against the eager ones. Sizes on both sides of each limit: blocks that leave a remainder of a wave's
ten, of a workgroup's forty, four tens a wave (from 327,680 blocks on) and 131,072 dofs."""
import numpy as np
import pytest

from tests.helpers import build_lattice

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mc():
    import muscade_amd
    return muscade_amd


def info(mc, out):
    v = np.zeros(7, np.int64)
    out.ctx.check(mc.lib.mh_get_scatter(out.ctx.h, mc._lib.i64ptr(v)), "scatter")
    return dict(zip(("nodes", "blocks", "rest", "tens", "joined", "long", "rlong"), v.tolist()))


def chain(mc, n):
    from muscade_amd.workloads import catenary_chains
    model, st = catenary_chains(nchain=1, nmin=n, nmax=n, seed=n)
    st.time = 1.0
    return model, st


def bits(a):
    return a.view(np.uint64)


def same_as_segmented(mc, model, st, OX, missions=("iter", "step")):
    """The eager and the graphed assembly, bitwise the same as the segmented scatter's."""
    outs = [mc.AssemblySweepX(OX, model, st.dis, graph=g) for g in (False, True, False)]
    if OX:
        for o in outs:
            o.c = mc.Newmarkβcoefficients(OX, 0.05)
    i = info(mc, outs[1])
    outs[2].ctx.check(mc.lib.mh_set_scatter_variant(outs[2].ctx.h, 3), "variant")
    assert info(mc, outs[2])["nodes"] == 0
    for mission in missions:
        ref = [x.copy() for x in outs[2].assemble(st, mission)]
        for o in outs[:2]:
            for _ in range(2):
                r, k = o.assemble(st, mission)
                assert np.array_equal(bits(r), bits(ref[0])) and np.array_equal(bits(k), bits(ref[1])), (mission, o.graph)
    return i


@pytest.mark.parametrize("n", list(range(1, 14)) + [39, 40, 41, 400])
def test_chains_by_nodes(mc, n):
    print("case", n, flush=True)
    model, st = chain(mc, n)
    i = same_as_segmented(mc, model, st, 1 + n % 2)
    # the inner nodes' three blocks; the anchor's columns carry λ rows, the top's first has its load's entry,
    # and their 153 nz outweigh the blocks below n = 3
    assert (i["blocks"], i["nodes"], i["joined"], i["tens"]) == (3 * n - 3, n >= 3, n >= 3, n >= 3), i


def test_lattice_by_nodes_and_compact(mc):
    model, st = build_lattice(6, 7, 5, seed=3)
    st = st.copy().with_ders(1, 3, 1)
    i = same_as_segmented(mc, model, st, 2)
    assert i["nodes"] == 1 and i["joined"] == 1, i
    i = same_as_segmented(mc, model, st, 0, ("iter",))     # compact matrices stay with the segmented scatter
    assert i["nodes"] == 0 and i["joined"] == 0, i


def test_bars_stay_segmented(mc):
    from tests.test_chain_layout import bar_chain, random_state
    model = bar_chain(n=11)
    i = same_as_segmented(mc, model, random_state(model, 2, scale=1e-2), 2)
    assert i["nodes"] == 0 and i["blocks"] == 0, i


@pytest.mark.parametrize("n,tens,joined", [(21_840, 1, 1), (21_850, 1, 0), (109_220, 1, 0), (109_250, 4, 0), (109_257, 4, 0)])
def test_limits(mc, n, tens, joined):
    print("case", n, flush=True)
    model, st = chain(mc, n)
    i = same_as_segmented(mc, model, st, 2)
    assert (i["nodes"], i["tens"], i["joined"]) == (1, tens, joined), i


@pytest.mark.parametrize("n", [50, 21_840, 21_850, 109_257])
def test_newton_iteration_into_the_blocks(mc, n):
    from muscade_amd.chainsolve import ChainSolver
    print("case", n, flush=True)
    model, st = chain(mc, n)
    c = mc.Newmarkβcoefficients(2, 0.05)
    states = []
    for graph in (False, True):
        out = mc.AssemblySweepX(2, model, st.dis, graph=graph)
        out.c = c
        cs = ChainSolver(out)
        out.set_state(st, st.time)
        norms = []
        for k in range(4):
            if graph:
                norms.append(cs.iteration_graph(2, k == 0, c.array()))
            else:
                out.assemble(st, "step" if k == 0 else "iter", fetch=False, upload=False)
                cs.solve()
                norms.append(cs.newton_update(2, k == 0, c.array()))
        end = st.copy()
        cs.fetch_X(end, 2)
        states.append((norms, end.X))
    assert states[0][0] == states[1][0]
    for a, b in zip(states[0][1], states[1][1]):
        assert np.array_equal(bits(a), bits(b))


def test_tuning_on_request(mc):
    """Where the nz go by nodes the segmented shapes are timed when they are asked for, beside the
    assembled values and the times of the last assembly; a shape that was set stays."""
    import ctypes
    model, st = chain(mc, 400)
    out = mc.AssemblySweepX(2, model, st.dis)
    out.c = mc.Newmarkβcoefficients(2, 0.05)
    out.assemble(st, "iter")
    before, times = out.nzval.copy(), out.timings()
    for variant in (None, 5):
        if variant is not None:
            out.ctx.check(mc.lib.mh_set_scatter_variant(out.ctx.h, variant), "variant")
        v, ms = ctypes.c_int(), (ctypes.c_float * 16)()
        out.ctx.check(mc.lib.mh_get_tuning(out.ctx.h, ctypes.byref(v), ms), "tuning")
        assert 0 <= v.value < 16 and all(x > 0 for x in ms) and variant in (None, v.value)
        out.ctx.check(mc.lib.mh_get_nzval(out.ctx.h, mc._lib.dptr(out.nzval)), "nzval")
        assert np.array_equal(bits(out.nzval), bits(before)) and np.array_equal(out.timings(), times)
        assert info(mc, out)["nodes"] == (variant is None)
