"""The gradient pass and the fold of batches over rows and tiles: gradients of
every instance against the labels (a cut arc leads from the source side to the
sink side inside the grid), through the per-instance and the all-instances call
and into device tensors off any vector alignment, at row lengths around the 4
nodes of a lane, the 32 of a tile and the 256 of a wave; flows and labels of the
same batches, whose capacities are folded tile by tile, against the oracle."""
import numpy as np
import pytest

import oracle_lib as ol
from conftest import random_grid

pytestmark = pytest.mark.gpu

BATCHES = [
    [(n, 5, 1, c) for n in (1, 2, 3, 4, 5, 6, 7) for c in (4, 8)],
    [(31, 9, 1, 8), (32, 8, 1, 4), (33, 1, 1, 8), (64, 3, 1, 4), (1, 70, 1, 8)],
    [(255, 6, 1, 4), (256, 5, 1, 4), (257, 4, 1, 4)],
    [(1025, 3, 1, 8), (20, 40, 1, 8)],
    [(300, 37, 1, 8)],
    [(5, 4, 3, 6), (33, 9, 2, 6), (8, 8, 4, 6), (260, 3, 3, 6)],
]


def gradients(lab, shape, dirs):
    nx, ny, nz, conn = shape
    lab = lab.reshape(nz, ny, nx)
    z, y, x = np.mgrid[:nz, :ny, :nx]
    out = []
    for dx, dy, dz in dirs[:conn]:
        X, Y, Z = x + dx, y + dy, z + dz
        inside = (X >= 0) & (X < nx) & (Y >= 0) & (Y < ny) & (Z >= 0) & (Z < nz)
        far = lab[np.clip(Z, 0, nz - 1), np.clip(Y, 0, ny - 1), np.clip(X, 0, nx - 1)]
        out.append((inside & (lab == 1) & (far == 0)).astype(np.float32).ravel())
    return np.array(out)


@pytest.mark.parametrize("batch", BATCHES, ids=lambda b: f"{len(b)}x{b[0][0]}-{b[0][3]}c")
@pytest.mark.parametrize("relabel", [0, 1])
def test_batch_gradients_gpu(gpu, batch, relabel):
    import torch
    rng = np.random.default_rng(sum(s[0] for s in batch))
    g = gpu.GridGraph(batch)
    want = []
    for i, (nx, ny, nz, conn) in enumerate(batch):
        cs, ct, caps = random_grid(rng, nx, ny, nz, conn)
        cs[0] += 1
        want.append(ol.maxflow(nx, ny, nz, conn, cs, ct, caps)[:2])
        g.set_terminal_caps(cs, ct, inst=i)
        g.set_all_neighbor_caps(caps, inst=i)
    print("case batch gradients", batch, relabel, flush=True)
    for _ in range(3):  # masks built, built and kept, copied
        assert g.solve(initial_relabel=relabel).converged == 1
        for i, (f, l) in enumerate(want):
            assert g.flow(inst=i) == f and np.array_equal(g.labels(inst=i), l)
    dcs, dct, dnb = g.backward_all()
    at = 0
    for i, shape in enumerate(batch):
        n, conn, lab = want[i][1].size, shape[3], want[i][1]
        dirs = gpu.DIRS_3D if conn == 6 else gpu.DIRS_2D
        ref = gradients(lab, shape, dirs)
        assert np.array_equal(dcs[at:at + n], (lab == 0).astype(np.float32))
        assert np.array_equal(dct[at:at + n], (lab == 1).astype(np.float32))
        assert np.array_equal(dnb[:conn, at:at + n], ref)
        at += n
        a, b, c = g.backward(i)
        assert np.array_equal(a, (lab == 0).astype(np.float32))
        assert np.array_equal(b, (lab == 1).astype(np.float32))
        assert np.array_equal(c, ref)
        t = [torch.full((k * n + 2,), -1.0, device="cuda") for k in (1, 1, conn)]
        v = [q[1:-1] for q in t]
        g.backward(i, out=(v[0], v[1], v[2].view(conn, n)))
        torch.cuda.synchronize()
        assert np.array_equal(v[1].cpu().numpy(), b) and np.array_equal(v[0].cpu().numpy(), a)
        assert np.array_equal(v[2].cpu().numpy().reshape(conn, n), c)
        assert all(float(q[0]) == -1 and float(q[-1]) == -1 for q in t)
    g.close()


@pytest.mark.parametrize("batch", [
    [(1, 40000, 1, 8)], [(3, 9000, 1, 4)], [(124, 70, 1, 8)], [(128, 67, 1, 4)], [(129, 40, 1, 8)],
    [(5, 40, 90, 6)], [(126, 9, 7, 6)], [(20000, 1, 1, 8)],
    [(16, 16, 1, 8)] * 30 + [(1, 3, 1, 4)] * 9, [(128, 5, 1, 8), (129, 5, 1, 4), (2, 60, 1, 8)] * 3,
], ids=lambda b: f"{len(b)}x{b[0][0]}-{b[0][3]}c")
def test_short_rows_gradients_gpu(gpu, batch):
    """Rows that a wave takes several of at once: lengths up to and past the 128
    nodes where it does, many rows per wave, instances that begin inside a wave's
    rows, and one row that many waves share."""
    rng = np.random.default_rng(len(batch) + batch[0][0])
    g = gpu.GridGraph(batch)
    labs = []
    for i, (nx, ny, nz, conn) in enumerate(batch):
        cs, ct, caps = random_grid(rng, nx, ny, nz, conn)
        cs[0] += 1
        labs.append(ol.maxflow(nx, ny, nz, conn, cs, ct, caps)[1])
        g.set_terminal_caps(cs, ct, inst=i)
        g.set_all_neighbor_caps(caps, inst=i)
    print("case short rows", batch[0], len(batch), flush=True)
    assert g.solve().converged == 1
    dcs, dct, dnb = g.backward_all()
    at = 0
    for i, shape in enumerate(batch):
        n, conn, lab = labs[i].size, shape[3], labs[i]
        ref = gradients(lab, shape, gpu.DIRS_3D if conn == 6 else gpu.DIRS_2D)
        assert np.array_equal(dcs[at:at + n], (lab == 0).astype(np.float32))
        assert np.array_equal(dct[at:at + n], (lab == 1).astype(np.float32))
        assert np.array_equal(dnb[:conn, at:at + n], ref)
        at += n
        a, b, c = g.backward(i)
        assert np.array_equal(a, (lab == 0).astype(np.float32))
        assert np.array_equal(b, (lab == 1).astype(np.float32))
        assert np.array_equal(c, ref)
    g.close()
