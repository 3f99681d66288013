"""Dynamic beams at the edges of the device's tiles of 64 elements: :step and :iter assembly, the
adjoint and the direct step, with random, equal and exactly zero node rotations, against the
oracle. Normwise relative error ≤ 1e-12, the bound of the other element tests."""
import numpy as np
import pytest

from tests.helpers import oracle_model, relerr
from tests.test_gpu_direct import add_supports, compare
from tests.test_gpu_dynamic import DT, dyn_beams
from tests.test_gpu_vjp import check, oracle_vjp

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.fixture(scope="module")
def mc():
    import muscade_amd
    return muscade_amd


def beams(mc, n, OX, rotation, udof):
    model, state, *rest = dyn_beams(mc, n, seed=1000 * OX + n, rotscale=0. if rotation == "zero" else 0.4, udof=udof)
    if rotation == "equal":
        d = state.dis.dis[0].X - 1
        for x in state.X:
            x[d[:, 9:12]] = x[d[:, 3:6]]
    return model, state, rest


@pytest.mark.parametrize("OX", [1, 2])
@pytest.mark.parametrize("n,rotation", [(1, "random"), (63, "random"), (64, "random"), (65, "random"), (129, "random"),
                                        (65, "equal"), (65, "zero")])
def test_tile_edges(mc, OX, n, rotation):
    print("case", OX, n, rotation, flush=True)
    udof = n % 2 == 0
    model, state, rest = beams(mc, n, OX, rotation, udof)
    out = mc.AssemblySweepX(OX, model, state.dis)
    out.c = mc.Newmarkβcoefficients(OX, DT, 0.25, 0.5)
    om = oracle_model(model, state.dis)
    for mission in ("step", "iter"):
        Lλ, nzval = out.assemble(state, mission)
        r, rhs, nz, err = om.assemble(OX, 0 if mission == "step" else 1, out.c.array(), state.X[:OX + 1],
                                      state.U[0] if udof else None, None)
        assert r == 0, err
        assert relerr(Lλ, rhs) <= TOL and relerr(nzval, nz) <= TOL, mission
    lam = np.random.default_rng(n).normal(size=model.ndof["X"])
    gX, gU, _ = out.vjp(state, lam, OX=OX)
    check(gX, gU, oracle_vjp(model, state, lam, OX, None))
    if n > 1:
        model.locked = False
        add_supports(mc, model, list(range(1, 2 * n + 1)), np.random.default_rng(0))
        s2 = mc.initialize(model, nXder=3, time=0.7)
        for k in range(3):
            s2.X[k][:state.X[k].size] = state.X[k]
        if udof:
            s2.U[0][:] = state.U[0]
        compare(mc, model, s2, np.random.default_rng(1).normal(size=model.ndof["X"]), OX, 0)
