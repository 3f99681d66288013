"""Static beams at the edges of the device's tiles (64 elements a wave), with zero, tiny, equal and
large node rotations: Lλ, Lλx and the adjoint against the oracle. Normwise relative error ≤ 1e-12,
the bound of the other element tests."""
import numpy as np
import pytest

from tests.helpers import oracle_model, relerr
from tests.test_gpu_dynamic import dyn_beams
from tests.test_gpu_vjp import check, oracle_vjp

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.fixture(scope="module")
def mc():
    import muscade_amd
    return muscade_amd


@pytest.mark.parametrize("n,rotscale", [(1, 0.4), (63, 0.4), (64, 0.4), (65, 0.4), (129, 0.4), (65, 0.), (65, 1e-8),
                                        (65, 1.2), (65, "equal")])
def test_static_tile_edges(mc, n, rotscale):
    print("case", n, rotscale, flush=True)
    udof = n % 2 == 0
    model, state, *_ = dyn_beams(mc, n, seed=500 + n, rotscale=0.4 if rotscale == "equal" else rotscale, udof=udof)
    if rotscale == "equal":
        d = state.dis.dis[0].X - 1
        state.X[0][d[:, 9:12]] = state.X[0][d[:, 3:6]]
    out = mc.AssemblySweepX(0, model, state.dis)
    Lλ, nzval = out.assemble(state, "iter")
    om = oracle_model(model, state.dis)
    r, rhs, nz, err = om.assemble(0, 1, out.c.array(), state.X[:1], state.U[0] if udof else None, None)
    assert r == 0, err
    assert relerr(Lλ, rhs) <= TOL and relerr(nzval, nz) <= TOL
    lam = np.random.default_rng(n).normal(size=model.ndof["X"])
    gX, gU, _ = out.vjp(state, lam, OX=0)
    check(gX, gU, oracle_vjp(model, state, lam, 0, None))
