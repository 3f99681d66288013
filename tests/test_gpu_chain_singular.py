"""Which diagonal block a failed chain solve names: of those with a zero pivot the one of the earliest
level of the reduction, and of a level the first in chain order, wherever the blocks' workgroups run
(64 blocks each, hundreds at a time) and in every solve. A node whose rows and columns are zero has a
zero pivot at its block's level and leaves its neighbours alone."""
import ctypes
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mc():
    import muscade_amd
    return muscade_amd


CASES = [(3000, [1], 1), (3000, [0], 0), (3000, [2999, 64, 32], 2999), (3000, [0, 2944], 2944),
         (9000, [4096, 448 + 32, 64], 448 + 32),
         (200000, [32, 64 * 3000 + 1], 64 * 3000 + 1),    # the first chunk is done before the last one starts
         (200000, [64 * 3000 + 1, 64 * 2 + 1, 64 * 2 + 2], 64 * 2 + 1),
         (200000, [64 * 64 * 40, 64 * 64 * 2 + 64], 64 * 64 * 2 + 64)]


@pytest.mark.parametrize("nblock,bad,named", CASES)
def test_first_block_of_the_earliest_level(mc, nblock, bad, named):
    from muscade_amd.chainsolve import ChainSolver
    from muscade_amd.workloads import catenary_chains
    print("case", nblock, bad, flush=True)
    model, st = catenary_chains(nchain=1, nmin=nblock - 1, nmax=nblock - 1, seed=1, disp=1e-5, rot=1e-5)
    st.time = 1.0
    out = mc.AssemblySweepX(2, model, st.dis)
    out.c = mc.Newmarkβcoefficients(2, 0.05)
    out.assemble(st, "iter")
    cs = ChainSolver(out)
    assert cs.layout.nblock == nblock
    node = np.asarray(model.dofnode("X"))
    nodes = [cs.layout.node_order[b] for b in bad]
    dead = np.isin(node, nodes) & (np.arange(out.nX) < 6 * nblock)
    col = np.repeat(np.arange(out.nX), np.diff(out.colptr))
    row = out.rowval - 1
    # a node's own dofs, not the multipliers of its supports (whose couplings stay)
    mult = np.zeros(out.nX, bool)
    mult[[i for i, p in enumerate(cs.layout.pos) if p < 0]] = True
    out.nzval[(dead[col] | dead[row]) & ~mult[col] & ~mult[row]] = 0.
    k = ctypes.POINTER(ctypes.c_double)()
    out.ctx.check(mc.lib.mh_device_outputs(out.ctx.h, None, ctypes.byref(k)), "outputs")
    to_device = 1
    assert ctypes.CDLL("libamdhip64.so.7").hipMemcpy(k, out.nzval.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(out.nzval.nbytes),
                                                   to_device) == 0
    for _ in range(4):
        with pytest.raises(mc.MuscadeError) as e:
            cs.solve()
        reason = e.value.dbg["reason"]
        assert int(re.search(r"diagonal block (\d+)", reason).group(1)) == named, reason
        level = "the last block" if named == 0 else f"reduction level {named & -named})"
        assert level in reason, reason
