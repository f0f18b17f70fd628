"""The device's decision when to relabel: work, not visits alone.  A few nodes
that hand a unit of excess around, cut off from every deficit, keep one tile
active and count one visit a sweep; without the stall test, only the cost of such
sweeps ends them.  Flows and labels against the oracle, bit-exact."""
import numpy as np
import pytest

import oracle_lib as ol
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


def noisy_object(nx, ny, conn, seed):
    """Unaries of a noisy disc and contrast-weighted arcs, as flat int32."""
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:ny, 0:nx]
    inside = ((y - 0.5 * ny) / (0.3 * ny)) ** 2 + ((x - 0.5 * nx) / (0.35 * nx)) ** 2 < 1
    grey = np.where(inside, 170.0, 90.0) + rng.normal(0, 30, (ny, nx))
    logit = np.rint((grey - 130.0) * 0.8).astype(np.int32)
    caps = np.zeros((conn, ny, nx), np.int32)
    for d, (dx, dy) in enumerate([(1, 0), (-1, 0), (0, 1), (0, -1), (1, 1), (-1, -1), (-1, 1),
                                  (1, -1)][:conn]):
        far = np.full((ny, nx), np.inf)
        far[max(0, -dy):ny - max(0, dy), max(0, -dx):nx - max(0, dx)] = \
            grey[max(0, dy):ny - max(0, -dy), max(0, dx):nx - max(0, -dx)]
        lam = 50.0 if d < 4 else 35.36
        caps[d] = np.rint(lam * np.exp(-(far - grey) ** 2 / 4050.0))
    return np.maximum(logit, 0).ravel(), np.maximum(-logit, 0).ravel(), caps.reshape(conn, -1)


@pytest.mark.parametrize("nx,ny,conn", [(1000, 1000, 4), (960, 900, 4), (1500, 1100, 8)])
def test_without_the_stall_test_gpu(gpu, nx, ny, conn):
    for seed in range(3):
        cs, ct, caps = noisy_object(nx, ny, conn, seed)
        f, l, ok = ol.maxflow(nx, ny, 1, conn, cs, ct, caps)
        g = gpu.GridGraph([(nx, ny, 1, conn)])
        g.set_terminal_caps(cs, ct)
        g.set_all_neighbor_caps(caps)
        say("case without the stall test", nx, ny, conn, seed)
        st = g.solve(stall_ratio=0.0)
        assert st.converged == 1 and g.flow() == f
        assert np.array_equal(g.labels(), l)
        assert st.sweeps < 500, st.sweeps
        g.close()
