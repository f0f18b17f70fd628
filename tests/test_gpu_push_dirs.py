"""The push kernel's choice of 4 or 8 directions and of its visit caps: flows
and labels against the oracle for one-instance and batched graphs whose
instances are all 4-connected, all 8-connected or mixed, at the edges of every
2D tile shape, and under caps below, at and above each other.  Bit-exact."""
import numpy as np
import pytest

import oracle_lib as ol
from conftest import random_grid
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (15, 17), (31, 8), (33, 9), (64, 4), (65, 33), (100, 47)]
CAPS = [dict(), dict(max_local_iters=1, sparse_local_iters=3),
        dict(max_local_iters=3, sparse_local_iters=1),
        dict(max_local_iters=1000, sparse_local_iters=1 << 30), dict(sparse_local_iters=-1)]


@pytest.mark.parametrize("tile", ["32x8", "64x4", "16x16"])
@pytest.mark.parametrize("conns", [(4,), (8,), (4, 4, 4), (8, 8), (4, 8, 4)])
def test_push_directions_gpu(gpu, conns, tile):
    rng = np.random.default_rng(sum(conns) * 10 + len(conns))
    for first in range(len(SIZES)):
        shapes = [SIZES[(first + 2 * k) % len(SIZES)] + (1, c) for k, c in enumerate(conns)]
        g = gpu.GridGraph(shapes)
        want = []
        for k, (nx, ny, nz, conn) in enumerate(shapes):
            cs, ct, caps = random_grid(rng, nx, ny, nz, conn)
            cs[0] += 1
            want.append(ol.maxflow(nx, ny, nz, conn, cs, ct, caps)[:2])
            g.set_terminal_caps(cs, ct, inst=k)
            g.set_all_neighbor_caps(caps, inst=k)
        for opts in CAPS:
            say("case push directions", shapes, tile, opts)
            assert g.solve(tile_shape=tile, **opts).converged == 1
            for k, (f, l) in enumerate(want):
                assert g.flow(inst=k) == f
                assert np.array_equal(g.labels(inst=k), l)
        g.close()


@pytest.mark.parametrize("conn,shape", [(8, (1500, 1100)), (6, (96, 96, 110))])
def test_cap_of_sparse_launches_past_the_grid_gpu(gpu, conn, shape):
    """Colour classes of more tiles than workgroups of a push launch that takes
    its tiles from the flags: its visits go up to the cap of sparse launches, as
    those of smaller classes do."""
    nx, ny, nz = shape + (1,) * (3 - len(shape))
    rng = np.random.default_rng(0)
    cs, ct, caps = random_grid(rng, nx, ny, nz, conn, term_max=3, seed_frac=0.001)
    g = gpu.GridGraph([(nx, ny, nz, conn)])
    g.set_terminal_caps(cs, ct)
    g.set_all_neighbor_caps(caps)
    print("case cap of sparse launches", shape, conn, flush=True)
    for cap in (2, 16):
        st = g.solve(max_local_iters=2, sparse_local_iters=cap, initial_relabel=1, max_sweeps=8)
        per_visit = st.local_iters / st.push_tiles
        assert per_visit <= 2 if cap == 2 else per_visit > 3, (cap, per_visit)
    g.close()
