"""The global relabel on bit-parallel regions (64x64 nodes in 2D, 64x8x8 in
3D): flows and labels against the oracle on grids at the edges of a region --
one node, one column or row short of, equal to and past a region, several
regions with ragged ends -- and on a single corridor whose distances span more
than a region's 12-bit counts keep.  Every solve relabels first, so a distance
that is off strands excess or leaves it active.  Bit-exact."""
import numpy as np
import pytest

import oracle_lib as ol
from conftest import random_grid
from test_gpu_parity import say, serpentine, solve_grid

pytestmark = pytest.mark.gpu

SHAPES_2D = [(1, 1), (1, 130), (130, 1), (63, 64), (64, 64), (65, 63), (64, 65), (129, 200),
             (257, 66)]
SHAPES_3D = [(64, 8, 8), (63, 7, 9), (65, 9, 2), (1, 17, 16), (130, 8, 17), (20, 33, 40)]


@pytest.mark.parametrize("conn,shape", [(c, s + (1,)) for c in (4, 8) for s in SHAPES_2D]
                         + [(6, s) for s in SHAPES_3D])
def test_region_edges_gpu(gpu, conn, shape):
    nx, ny, nz = shape
    rng = np.random.default_rng(1000 * conn + 31 * nx + 7 * ny + nz)
    for frac in (0.002, 0.2):
        # few terminals: distances cross regions; many: most regions hold both
        cs, ct, caps = random_grid(rng, nx, ny, nz, conn, term_max=20, seed_frac=0.01)
        on = rng.random(cs.size) < frac
        on[0] = on[-1] = True
        cs, ct = np.where(on, cs, 0).astype(np.int32), np.where(on, ct, 0).astype(np.int32)
        cs[0], ct[-1] = 500, 700
        f, l, ok = ol.maxflow(nx, ny, nz, conn, cs, ct, caps)
        say("case region edges", conn, shape, frac)
        for opts in (dict(), dict(tile_shape="32x4x2" if nz > 1 else "64x4")):
            g, st = solve_grid(gpu, nx, ny, nz, conn, cs, ct, caps, initial_relabel=1, **opts)
            assert st.converged == 1
            assert g.flow() == f
            assert np.array_equal(g.labels(), l)
            g.close()


@pytest.mark.parametrize("shape", [(200, 203, 1), (70, 31, 9)])
def test_long_corridor_gpu(gpu, shape):
    nx, ny, nz = shape
    cs, ct, caps, conn = serpentine(nx, ny, nz)
    end = int(np.argmax(ct))
    ct[:] = 0
    ct[end] = 1000
    f, l, ok = ol.maxflow(nx, ny, nz, conn, cs, ct, caps)
    say("case long corridor", shape)
    g, st = solve_grid(gpu, nx, ny, nz, conn, cs, ct, caps, initial_relabel=1)
    assert st.converged == 1
    assert g.flow() == f
    assert np.array_equal(g.labels(), l)
    g.close()


@pytest.mark.parametrize("shape", [s + (1,) for s in SHAPES_2D] + SHAPES_3D)
def test_region_edges_tag_gpu(gpu, shape):
    """The tag flood over the regions: seeds on and off the source side, at the
    corners and inside, on a cut of dense terminals (many small components)."""
    nx, ny, nz = shape
    conn = 6 if nz > 1 else 8
    rng = np.random.default_rng(31 * nx + 7 * ny + nz)
    cs, ct, caps = random_grid(rng, nx, ny, nz, conn, cap_max=8)
    cs[0], ct[-1] = 500, 700
    say("case region edges tag", shape)
    g, st = solve_grid(gpu, nx, ny, nz, conn, cs, ct, caps)
    assert st.converged == 1
    lab = g.labels()
    for frac in (0.0, 0.02, 0.3):
        fg = (rng.random(nx * ny * nz) < frac).astype(np.uint8)
        fg[0] = fg[-1] = 1
        assert np.array_equal(g.tags(fg), ol.tag(nx, ny, nz, fg, lab))
    g.close()


@pytest.mark.parametrize("conn,shape", [(8, (300, 217, 1)), (4, (2100, 1100, 1)), (6, (70, 41, 33)),
                                        (6, (300, 190, 70))])
def test_relabel_gives_up_waiting_gpu(gpu, conn, shape):
    """A relabel whose waves give up waiting at once is finished by passes: one
    launch for everything (up to 512 regions) and above."""
    import ctypes
    nx, ny, nz = shape
    rng = np.random.default_rng(nx)
    cs, ct, caps = random_grid(rng, nx, ny, nz, conn, term_max=20, seed_frac=0.001)
    f, l, ok = ol.maxflow(nx, ny, nz, conn, cs, ct, caps)
    g = gpu.GridGraph([(nx, ny, nz, conn)])
    g.set_terminal_caps(cs, ct)
    g.set_all_neighbor_caps(caps)
    for ticks in (0, 1 << 22, 0):
        say("case relabel wait", conn, shape, ticks)
        assert gpu.lib().jfc_debug_relabel_wait(g._h, ctypes.c_int64(ticks)) == 0
        st = g.solve(initial_relabel=1)
        assert st.converged == 1 and st.global_relabels >= 1
        assert g.flow() == f
        assert np.array_equal(g.labels(), l)
    g.close()


@pytest.mark.parametrize("conn,shape", [(8, (300, 217, 1)), (4, (2100, 1100, 1)), (6, (70, 41, 33)),
                                        (6, (300, 190, 70))])
def test_tag_gives_up_waiting_gpu(gpu, conn, shape):
    """A tag flood whose waves give up waiting at once is finished by passes:
    one launch for everything (up to 512 regions) and above."""
    import ctypes
    nx, ny, nz = shape
    rng = np.random.default_rng(ny)
    cs, ct, caps = random_grid(rng, nx, ny, nz, conn, term_max=20, seed_frac=0.001)
    g, st = solve_grid(gpu, nx, ny, nz, conn, cs, ct, caps)
    assert st.converged == 1
    lab = g.labels()
    fg = (rng.random(nx * ny * nz) < 0.001).astype(np.uint8)
    fg[0] = 1
    want = ol.tag(nx, ny, nz, fg, lab)
    for ticks in (0, 1 << 22, 0):
        say("case tag wait", conn, shape, ticks)
        assert gpu.lib().jfc_debug_relabel_wait(g._h, ctypes.c_int64(ticks)) == 0
        assert np.array_equal(g.tags(fg), want)
    g.close()
