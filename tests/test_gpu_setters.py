"""The capacity setters' one pass (copy, range check, arcs that leave the
grid): planes read back from the graph equal the arrays given, with the
leaving arcs 0, at row lengths around the 64 lanes and 256 columns of a
workgroup, from host arrays, device tensors and device tensors that start off
any vector alignment; a single value past the range at either end of a plane
is refused, by the name of its plane, and leaves that plane zeroed."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1, 4), (31, 5, 1, 8), (32, 4, 1, 4), (63, 3, 1, 8), (65, 9, 1, 4), (255, 2, 1, 8),
          (256, 7, 1, 4), (257, 6, 1, 8), (1, 40, 1, 8), (520, 3, 1, 4), (33, 5, 3, 6),
          (64, 8, 8, 6), (7, 6, 2, 6)]


def steps(conn):
    if conn == 6:
        return [(1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)]
    return [(1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (1, 1, 0), (-1, -1, 0), (-1, 1, 0),
            (1, -1, 0)][:conn]


def inside(nx, ny, nz, step):
    z, y, x = np.mgrid[:nz, :ny, :nx]
    x, y, z = x + step[0], y + step[1], z + step[2]
    return ((x >= 0) & (x < nx) & (y >= 0) & (y < ny) & (z >= 0) & (z < nz)).ravel()


def given(a, how):
    if how == "host":
        return a
    import torch
    t = torch.zeros(a.size + 1, dtype=torch.int32, device="cuda")
    v = t[1:] if how == "offset" else t[:-1]
    v.copy_(torch.from_numpy(a.astype(np.int32)))
    torch.cuda.synchronize()
    return v


def planes(gpu, g, n, conn):
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    cs, ct, c = np.empty(n, np.int32), np.empty(n, np.int32), np.empty((conn, n), np.int32)
    assert gpu.lib().jfc_get_terminal_caps(g._h, 0, p(cs), p(ct), 0) == 0
    for d in range(conn):
        assert gpu.lib().jfc_get_neighbor_caps(g._h, 0, d, p(c[d]), 0) == 0
    return cs, ct, c


@pytest.mark.parametrize("how", ["host", "device", "offset"])
@pytest.mark.parametrize("shape", SHAPES)
def test_setters_gpu(gpu, shape, how):
    nx, ny, nz, conn = shape
    n = nx * ny * nz
    rng = np.random.default_rng(n + conn)
    top = 1 << 30
    cs, ct = (rng.integers(0, top + 1, n).astype(np.int32) for _ in range(2))
    caps = rng.integers(0, (1 << 26) + 1, (conn, n)).astype(np.int32)
    ef = rng.integers(-top, top + 1, n).astype(np.int32)
    print("case setters", shape, how, flush=True)
    g = gpu.GridGraph([shape])
    g.set_terminal_caps(given(cs, how), given(ct, how))
    for d in range(conn):
        g.set_neighbor_caps(d, given(caps[d], how))
    want = [np.where(inside(nx, ny, nz, s), caps[d], 0) for d, s in enumerate(steps(conn))]
    a, b, c = planes(gpu, g, n, conn)
    assert np.array_equal(a, cs) and np.array_equal(b, ct) and np.array_equal(c, want)
    g.set_excess(given(ef, how))
    a, b, _ = planes(gpu, g, n, conn)
    assert np.array_equal(a, np.maximum(ef, 0)) and np.array_equal(b, np.maximum(-ef, 0))
    for at in (0, n - 1):
        for lo, hi, plane in ((-1, top + 1, 0), (-1, top + 1, 1)):
            for v in (lo, hi, -(1 << 31)):
                x = [cs.copy(), ct.copy()]
                x[plane][at] = v
                with pytest.raises(gpu.JFCError) as err:
                    g.set_terminal_caps(given(x[0], how), given(x[1], how))
                assert ("source", "sink")[plane] in str(err.value)
                a, b, _ = planes(gpu, g, n, conn)
                assert not a.any() and not b.any()
        for v in (-top - 1, top + 1, -(1 << 31)):
            x = ef.copy()
            x[at] = v
            with pytest.raises(gpu.JFCError, match="excess"):
                g.set_excess(given(x, how))
        for v in (-1, (1 << 26) + 1):
            x = caps[0].copy()
            x[at] = v
            with pytest.raises(gpu.JFCError, match="neighbour"):
                g.set_neighbor_caps(0, given(x, how))
            _, _, c = planes(gpu, g, n, conn)
            assert not c[0].any() and np.array_equal(c[1:], want[1:])
    g.close()
