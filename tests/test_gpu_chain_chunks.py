"""The chain solve at the edges of its chunks: 64 blocks per workgroup, 128 in the last phase, one,
two and three phases, 6- and 3-dof blocks. Δx is a backward-stable solution (normwise backward
error ≤ 1e-14, the bound of the other chain solves) and a second solve repeats it bitwise."""
import numpy as np
import pytest

from tests.test_chain_layout import backward_error, bar_chain, random_state
from tests.test_gpu_chainsolve import device_solve

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mc():
    import muscade_amd
    return muscade_amd


@pytest.mark.parametrize("kind,nblock", [("beam", n) for n in (2, 3, 63, 64, 65, 127, 128, 129, 192, 193, 64 * 128,
                                                               64 * 128 + 1, 64 * 129 + 63)]
                         + [("bar", n) for n in (2, 64, 128, 129, 8193)])
def test_chunk_edges(mc, kind, nblock):
    from muscade_amd.workloads import catenary_chains
    print("case", kind, nblock, flush=True)
    if kind == "bar":
        model = bar_chain(n=nblock - 1)
        st = random_state(model, 2, scale=1e-4)
    else:
        model, st = catenary_chains(nchain=1, nmin=nblock - 1, nmax=nblock - 1, seed=nblock, disp=1e-5, rot=1e-5)
        st.time = 1.0
    out, cs, K, r, dx = device_solve(mc, model, st, 2, "step")
    assert cs.layout.nblock == nblock and cs.layout.B == (3 if kind == "bar" else 6)
    assert backward_error(K, dx, r) <= 1e-14
    cs.solve()
    assert np.array_equal(cs.dx().view(np.uint64), dx.view(np.uint64))
