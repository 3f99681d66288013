"""Dynamic beams at the edges of every kernel's tile: 64 elements for the value pass and the records, 42 for
the directions of :iter, the adjoint and the direct step, 32 for :step, whose fourth wave has the δr lanes
(a last tile of one element, one short of full, full, one over). :iter and :step, the adjoint and the
direct step of a single element and of each size against the oracle, normwise relative error ≤ 1e-12,
the bound of the other element tests."""
import numpy as np
import pytest

from tests.helpers import oracle_model, relerr
from tests.test_gpu_direct import add_supports, compare
from tests.test_gpu_dynamic import DT, dyn_beams
from tests.test_gpu_vjp import check, oracle_vjp

pytestmark = pytest.mark.gpu
TOL = 1e-12
VALUE, DIRECTION, STEP = 64, 42, 32
SIZES = sorted({1, 2} | {k * t + d for t in (VALUE, DIRECTION, STEP) for k in (1, 2) for d in (-1, 0, 1)})


@pytest.fixture(scope="module")
def mc():
    import muscade_amd
    return muscade_amd


@pytest.mark.parametrize("OX", [1, 2])
@pytest.mark.parametrize("n", SIZES)
def test_assembly_and_adjoint(mc, OX, n):
    print("case", OX, n, flush=True)
    udof = n % 2 == 1
    model, state, *_ = dyn_beams(mc, n, seed=2000 * OX + n, rotscale=0.4, udof=udof)
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


@pytest.mark.parametrize("OX", [0, 1, 2])
@pytest.mark.parametrize("n", SIZES)
def test_direct_step(mc, OX, n):
    print("case", OX, n, flush=True)
    udof = n % 2 == 1
    model, state, *_ = dyn_beams(mc, n, seed=3000 * OX + n, rotscale=0.4, udof=udof)
    model.locked = False
    add_supports(mc, model, list(range(1, 2 * n + 1)), np.random.default_rng(0))
    st = mc.initialize(model, nXder=3, time=0.7)
    for k in range(3):
        st.X[k][:state.X[k].size] = state.X[k]
    if udof:
        st.U[0][:] = state.U[0]
    compare(mc, model, st, np.random.default_rng(1).normal(size=model.ndof["X"]), OX, 0)
