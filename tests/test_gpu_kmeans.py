"""The k-means of the data term (jfc_model_image) against the oracle at the
seed counts where its device forms change -- one wave, one round of the
workgroup, the last round of the one-launch form and the first count past it,
different on the two sides -- for every feature type, cluster counts of 1 to
16, values over the whole range of the type and few distinct values (which
tie distances and leave clusters empty).  Centroids, iteration counts and unary
capacities, bit-exact."""
import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu

COUNTS = [(1, 2), (63, 64), (65, 1023), (1024, 1025), (2047, 4097), (7169, 8191), (8192, 8192),
          (8193, 20), (5, 12000)]


@pytest.mark.parametrize("counts", COUNTS, ids=lambda c: f"{c[0]}-{c[1]}")
@pytest.mark.parametrize("kind", ["rgb", "grey", "grey16"])
def test_kmeans_counts_gpu(gpu, kind, counts):
    nx, ny = 160, 130
    top = 65535 if kind == "grey16" else 255
    R = 1024 if kind == "grey16" else 255
    C = 3 if kind == "rgb" else 1
    dt = np.uint16 if kind == "grey16" else np.uint8
    rng = np.random.default_rng(sum(counts) + top + C)
    at = rng.permutation(nx * ny)
    sd = np.zeros(nx * ny, np.uint8)
    sd[at[:counts[0]]] = 1
    sd[at[counts[0]:sum(counts)]] = 2
    sd = sd.reshape(ny, nx)
    for k, distinct in ((1, 0), (2, 5), (5, 0), (8, 6), (16, 0), (11, 40)):
        img = rng.integers(0, top + 1, (ny, nx, C))
        if distinct:  # evenly spaced levels: midpoints are levels again
            img = img * distinct // (top + 1) * (top // (distinct - 1))
        else:
            img[0, 0], img[-1, -1] = 0, top
        img = img.astype(dt) if C == 3 else img[..., 0].astype(dt)
        print("case kmeans", kind, counts, k, distinct, flush=True)
        cs, ct, caps, info = ol.model_image(img, sd, 4, k=k, R=R)
        g = gpu.GridGraph([(nx, ny, 1, 4)])
        st = g.model_image(img, sd, k_fg=k, k_bg=k, rng=R)
        assert np.array_equal(np.array(st.centroids_fg[:k * C]), info["cfg"].ravel())
        assert np.array_equal(np.array(st.centroids_bg[:k * C]), info["cbg"].ravel())
        assert (st.iters_fg, st.iters_bg) == (info["iters_fg"], info["iters_bg"])
        gcs, gct = g.terminal_caps()
        assert np.array_equal(gcs, cs) and np.array_equal(gct, ct)
        g.close()
