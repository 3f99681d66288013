"""Adjoints of other orders than the one that was prepared, between assemblies eager and replayed: the
records of the dynamic beams grow to the highest order asked for, and every result is bitwise that of
a context of its own."""
import numpy as np
import pytest

from tests.test_gpu_dynamic import DT, dyn_beams

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mc():
    import muscade_amd
    return muscade_amd


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("n", [1, 64, 65, 200])
@pytest.mark.parametrize("OX", [0, 1, 2])
def test_orders(mc, OX, n, graph):
    print("case", OX, n, graph, flush=True)
    model, state, *_ = dyn_beams(mc, n, seed=n, rotscale=0.4, udof=n % 2 == 0)
    lam = np.random.default_rng(n).normal(size=model.ndof["X"])

    def context():
        out = mc.AssemblySweepX(OX, model, state.dis, graph=graph)
        out.c = mc.Newmarkβcoefficients(OX, DT)
        return out

    def assembled(out):
        return [np.concatenate([x.copy() for x in out.assemble(state, m)]) for m in ("iter", "step")]

    def gradient(out, k):
        gX, gU, _ = out.vjp(state, lam, OX=k)
        return np.concatenate([*gX, gU])

    ref = assembled(context())
    refs = [gradient(context(), k) for k in range(3)]
    out = context()
    for k in (None, 1, None, 0, 2, None, 1, 0, 2, None):
        got, want = (assembled(out), ref) if k is None else ([gradient(out, k)], [refs[k]])
        for a, b in zip(got, want):
            assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), k
