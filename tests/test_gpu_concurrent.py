"""One-launch searches (relabel, cut and tag floods) and what ends them: searches
longer than the time a wave waits.  Flows and labels against the oracle,
bit-exact."""
import ctypes

import numpy as np
import pytest

import oracle_lib as ol
from test_gpu_parity import say, serpentine

pytestmark = pytest.mark.gpu


def make(gpu, shape, cs, ct, caps, ticks=None):
    g = gpu.GridGraph([shape])
    g.set_terminal_caps(cs, ct)
    g.set_all_neighbor_caps(caps)
    if ticks is not None:
        assert gpu.lib().jfc_debug_relabel_wait(g._h, ctypes.c_int64(ticks)) == 0
    return g


@pytest.mark.parametrize("shape", [(64, 4001, 1), (70, 31, 9)])
def test_search_longer_than_the_wait_gpu(gpu, shape):
    """A relabel along one corridor takes 5-20 ms, its front in one region at a
    time; the other waves wait longer than the bound of 1 ms, and the search
    goes on as one launch."""
    nx, ny, nz = shape
    cs, ct, caps, conn = serpentine(nx, ny, nz)
    end = int(np.argmax(ct))
    ct[:] = 0
    ct[end] = 1000
    f, l, ok = ol.maxflow(nx, ny, nz, conn, cs, ct, caps)
    g = make(gpu, (nx, ny, nz, conn), cs, ct, caps, ticks=100_000)
    say("case search longer than the wait", shape)
    st = g.solve(initial_relabel=1)
    assert st.converged == 1 and g.flow() == f
    assert np.array_equal(g.labels(), l)
    assert st.relabel_passes == st.global_relabels
    g.close()
