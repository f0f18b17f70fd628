"""Searches (relabel, cut and tag floods) that take a launch per pass: from the
first pass on, as graphs with more regions than a one-launch search can look
after do, and after a one-launch search gave up waiting.  Grids at the edges of a
region, long corridors and uneven batches of both connectivities, whose
instances share the launches; flows, labels and tags against the oracle,
bit-exact."""
import ctypes

import numpy as np
import pytest

import oracle_lib as ol
from conftest import random_grid
from test_gpu_parity import say, serpentine

pytestmark = pytest.mark.gpu

WAYS = ["passes", "gives up"]


def take(gpu, g, way):
    L = gpu.lib()
    if way == "passes":
        assert L.jfc_debug_search_passes(g._h, 1) == 0
    else:
        assert L.jfc_debug_relabel_wait(g._h, ctypes.c_int64(0)) == 0


def check(gpu, shapes, graphs, way, seed=0, solves=2):
    rng = np.random.default_rng(seed)
    g = gpu.GridGraph(shapes)
    want = []
    for i, (s, (cs, ct, caps)) in enumerate(zip(shapes, graphs)):
        g.set_terminal_caps(cs, ct, inst=i)
        g.set_all_neighbor_caps(caps, inst=i)
        want.append(ol.maxflow(*s, cs, ct, caps))
    take(gpu, g, way)
    for _ in range(solves):
        st = g.solve(initial_relabel=1)
        assert st.converged == 1 and st.global_relabels >= 1
        if way == "passes":
            assert st.relabel_passes >= 4 * st.global_relabels  # first, last, and two between
        assert list(g.flows()) == [w[0] for w in want]
        for i, s in enumerate(shapes):
            lab = g.labels(inst=i)
            assert np.array_equal(lab, want[i][1]), i
            fg = (rng.random(lab.size) < 0.02).astype(np.uint8)
            fg[0] = 1
            assert np.array_equal(g.tags(fg, inst=i), ol.tag(*s[:3], fg, lab)), i
    g.close()


@pytest.mark.parametrize("way", WAYS)
@pytest.mark.parametrize("shape", [(1, 1, 1, 4), (64, 64, 1, 8), (65, 63, 1, 4), (129, 200, 1, 8),
                                   (1, 130, 1, 8), (63, 7, 9, 6), (65, 9, 2, 6), (130, 17, 17, 6),
                                   (1600, 1500, 1, 8), (200, 190, 70, 6)])
def test_one_grid_gpu(gpu, shape, way):
    nx, ny, nz, conn = shape
    rng = np.random.default_rng(nx + 7 * ny + nz)
    cs, ct, caps = random_grid(rng, *shape, term_max=20, seed_frac=0.01)
    on = rng.random(cs.size) < 0.1
    cs, ct = np.where(on, cs, 0).astype(np.int32), np.where(on, ct, 0).astype(np.int32)
    cs[0], ct[-1] = 500, 700
    say("case one grid", shape, way)
    check(gpu, [shape], [(cs, ct, caps)], way)


@pytest.mark.parametrize("way", WAYS)
@pytest.mark.parametrize("shape", [(200, 203, 1), (70, 31, 9)])
def test_corridor_gpu(gpu, shape, way):
    cs, ct, caps, conn = serpentine(*shape)
    end = int(np.argmax(ct))
    ct[:] = 0
    ct[end] = 1000
    say("case corridor", shape, way)
    check(gpu, [shape + (conn,)], [(cs, ct, caps)], way, solves=1)


@pytest.mark.parametrize("way", WAYS)
@pytest.mark.parametrize("d3", [False, True])
def test_uneven_batch_gpu(gpu, d3, way):
    rng = np.random.default_rng(40 + d3)
    if d3:
        shapes = [(nx, ny, nz, 6) for nx, ny, nz in
                  [(64, 8, 8), (70, 31, 9), (5, 6, 7), (130, 20, 3), (1, 1, 2), (63, 25, 33)]]
    else:
        shapes = [(nx, ny, 1, c) for nx, ny, c in
                  [(64, 64, 8), (130, 70, 4), (1, 1, 4), (300, 17, 8), (65, 129, 4), (7, 200, 8),
                   (33, 33, 4), (257, 190, 8)]]
    graphs = []
    for s in shapes:
        cs, ct, caps = random_grid(rng, *s, term_max=20, seed_frac=0.01)
        cs[0] += 100
        ct[-1] += 100
        graphs.append((cs, ct, caps))
    say("case uneven batch", d3, way)
    check(gpu, shapes, graphs, way)
