"""One-launch searches (relabel, cut and tag floods) beside other work: graphs
solved from several threads on streams of their own, whose searches hold each
other's places on the device, and searches longer than the time a wave waits.
Flows and labels against the oracle, bit-exact."""
import ctypes
import threading
import time

import numpy as np
import pytest

import oracle_lib as ol
from conftest import random_grid
from test_gpu_parity import say, serpentine

pytestmark = pytest.mark.gpu


def make(gpu, shape, cs, ct, caps, ticks=None):
    g = gpu.GridGraph([shape])
    g.set_terminal_caps(cs, ct)
    g.set_all_neighbor_caps(caps)
    if ticks is not None:
        assert gpu.lib().jfc_debug_relabel_wait(g._h, ctypes.c_int64(ticks)) == 0
    return g


@pytest.mark.parametrize("shape", [(96, 96, 96, 6), (1400, 1400, 1, 4)])
def test_graphs_solved_at_the_same_time_gpu(gpu, shape):
    """Three graphs from three threads.  A search that another one keeps from its
    places does not wait for them until the bound, here 2 seconds."""
    import torch
    work = []
    for seed in range(3):
        rng = np.random.default_rng(seed)
        cs, ct, caps = random_grid(rng, *shape, term_max=3, seed_frac=0.0005)
        g = make(gpu, shape, cs, ct, caps, ticks=200_000_000)
        s = torch.cuda.Stream()
        g.set_stream(s.cuda_stream)
        g.solve(initial_relabel=1)
        work.append((g, s, g.flow(), g.labels(), ol.maxflow(*shape, cs, ct, caps)))
    for g, s, f, l, want in work:
        assert f == want[0] and np.array_equal(l, want[1])
    slow, wrong = [], []

    def solve(g, f, l):
        for i in range(6):
            t = time.perf_counter()
            st = g.solve(initial_relabel=1)
            slow.append(time.perf_counter() - t)
            fg = np.zeros(l.size, np.uint8)
            fg[::31] = 1
            g.tags(fg)
            if not (st.converged == 1 and g.flow() == f and np.array_equal(g.labels(), l)):
                wrong.append(i)

    say("case graphs at the same time", shape)
    threads = [threading.Thread(target=solve, args=(g, f, l)) for g, s, f, l, _ in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    assert max(slow) < 2.0, slow
    for g, *_ in work:
        g.close()


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


def test_sweeps_do_not_depend_on_the_clock_gpu(gpu):
    """When a stall relabels is decided by work, not by time: relabels that take
    longer (a launch per pass) change no solve.  The graph's rows are chains of
    their own, each in one wave of its tiles, so its sweeps are the same in every
    run; a steady front moves along each."""
    nx, ny = 4000, 64
    rng = np.random.default_rng(5)
    caps = np.zeros((4, ny, nx), np.int32)
    caps[0, :, :-1] = rng.integers(40, 60, (ny, nx - 1))
    caps[1, :, 1:] = rng.integers(0, 60, (ny, nx - 1))
    cs, ct = np.zeros((2, ny, nx), np.int32)
    cs[:, 0] = rng.integers(20, 60, ny)
    ct[:, -1] = rng.integers(20, 60, ny)
    cs, ct, caps = cs.ravel(), ct.ravel(), caps.reshape(4, -1)
    f, l, ok = ol.maxflow(nx, ny, 1, 4, cs, ct, caps)
    g = make(gpu, (nx, ny, 1, 4), cs, ct, caps)
    seen, stopped = set(), set()
    for ticks in (2_000_000, 0, 2_000_000, 0):
        say("case sweeps and the clock", ticks)
        assert gpu.lib().jfc_debug_relabel_wait(g._h, ctypes.c_int64(ticks)) == 0
        st = g.solve(tile_shape="32x8")
        assert st.converged == 1 and g.flow() == f
        assert np.array_equal(g.labels(), l)
        seen.add((st.sweeps, st.global_relabels))
        for first in (0, 1):
            st = g.solve(tile_shape="32x8", max_sweeps=100, initial_relabel=first)
            assert st.converged == 0
            stopped.add((first, st.sweeps, st.global_relabels, g.flow(), g.labels().tobytes()))
    assert len(seen) == 1 and min(seen)[1] >= 3, seen
    assert len(stopped) == 2
    g.close()
