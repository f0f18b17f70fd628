"""The widget model's seed scan and k-means (jfc_model_widget) against the
oracle: every capacity, the iteration counts and the centroids, bit-exact, at
the sizes where a path begins or ends -- one seed, k at its limits and at the
edges of the kernel's cluster counts, pixels seeded on both sides, seed maps
that do not start at a multiple of four bytes, and more seeds than one
workgroup takes.  A side without seeds is refused and changes no plane."""
import numpy as np
import pytest

from test_gpu_widget_model import check, random_case, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [2, 8, 9, 16, 17, 32])
def test_cluster_counts_gpu(gpu, k):
    shape = (131, 67, 1)
    say("case widget k", k)
    rgba, fg, bg = random_case(shape, k)
    check(gpu, shape, rgba, fg, bg, dict(lazy=True, k=k, weight=(0.3, 0.5, 0.2, 0.1)), solve=False)


@pytest.mark.parametrize("lazy", [True, False])
def test_seed_maps_gpu(gpu, lazy):
    shape = (97, 45, 1)
    rgba, fg, bg = random_case(shape, 3)
    kw = dict(lazy=lazy, k=5, bk_terminal=0.7)
    one_f, one_b = np.zeros_like(fg), np.zeros_like(bg)
    one_f[-1], one_b[0] = 1, 255
    say("case widget one seed a side", lazy)
    check(gpu, shape, rgba, one_f, one_b, kw, solve=False)
    both = fg | bg
    say("case widget pixels seeded on both sides", lazy)
    check(gpu, shape, rgba, both, both, kw, solve=False)


@pytest.mark.parametrize("rows", [171, 172])  # 65,322 / 65,704 seeds a side
def test_many_seeds_gpu(gpu, rows):
    shape = (382, 400, 1)
    say("case widget many seeds", rows)
    rgba, fg, bg = random_case(shape, rows)
    fg = fg.reshape(400, 382)
    bg = bg.reshape(400, 382)
    fg[:], bg[:] = 0, 0
    fg[:rows] = 1
    bg[400 - rows:] = 3
    check(gpu, shape, rgba, fg.ravel(), bg.ravel(), dict(lazy=True, k=8, kmeans_iterations=6),
          solve=False)


def test_unaligned_seed_maps_gpu(gpu):
    import torch
    shape = (61, 33, 1)
    n = shape[0] * shape[1]
    rgba, fg, bg = random_case(shape, 7)
    g = gpu.GridGraph([shape + (4,)])
    g.model_widget(rgba, fg, bg, k=6)
    want = g.terminal_caps() + (g.neighbor_caps(),)
    for off in (1, 2, 3):
        say("case widget unaligned", off)
        pad = torch.zeros(2, n + 8, dtype=torch.uint8, device="cuda")
        pad[0, off:off + n] = torch.from_numpy(fg).cuda()
        pad[1, off + 1:off + 1 + n] = torch.from_numpy(bg).cuda()
        h = gpu.GridGraph([shape + (4,)])
        h.model_widget(torch.from_numpy(rgba).cuda(), pad[0, off:off + n],
                       pad[1, off + 1:off + 1 + n], k=6)
        for a, b in zip(want, h.terminal_caps() + (h.neighbor_caps(),)):
            assert np.array_equal(a, b)
        h.close()
    g.close()


@pytest.mark.parametrize("lazy", [True, False])
def test_no_seeds_gpu(gpu, lazy):
    shape = (40, 30, 1)
    rgba, fg, bg = random_case(shape, 5)
    g = gpu.GridGraph([shape + (4,)])
    g.model_widget(rgba, fg, bg, lazy=lazy, k=3)
    want = g.terminal_caps() + (g.neighbor_caps(),)
    none = np.zeros_like(fg)
    for f, b in ((none, bg), (fg, none), (none, none)):
        say("case widget no seeds", lazy)
        with pytest.raises(gpu.JFCError) as e:
            g.model_widget(255 - rgba, f, b, lazy=lazy, k=3)
        assert e.value.code == gpu.ERR_NO_SEEDS
        for a, c in zip(want, g.terminal_caps() + (g.neighbor_caps(),)):
            assert np.array_equal(a, c)
    g.close()


@pytest.mark.parametrize("levels", [2, 3, 9])
@pytest.mark.parametrize("k", [8, 12])
def test_ties_gpu(gpu, k, levels):
    """Few grey levels: centroids that coincide, pixels on their centroid or
    halfway between two, clusters that empty."""
    shape = (67, 45, 1)
    say("case widget ties", levels, "clusters", k)
    rgba, fg, bg = random_case(shape, levels)
    rgba[:, :3] = (rgba[:, :1] % levels) * (255 // (levels - 1))
    rgba[:, 3] = 255
    check(gpu, shape, rgba, fg, bg, dict(lazy=True, k=k), solve=False)


def test_weights_without_a_norm_gpu(gpu):
    """Weights whose squares underflow normalise to infinity, and a 0 beside them
    to no number.  A movement that is no number does not count, so one such
    weight ends the k-means with its first assignment; with four, the clusters
    but the first empty, and a byte that no member has adds nothing to a mean."""
    shape = (67, 45, 1)
    rgba, fg, bg = random_case(shape, 4)
    rgba = np.maximum(rgba, 1)
    g = gpu.GridGraph([shape + (4,)])
    for n, its in ((1, 1), (4, 2)):
        say("case widget weights without a norm", n)
        st = g.model_widget(rgba, fg, bg, lazy=True, k=5, weight=[1e-30] * n + [0.0] * (4 - n))
        assert list(st.iterations) == [its, its]
        cent = np.ctypeslib.as_array(st.centroids)[:, :5]
        if n == 1:
            assert np.isposinf(cent[..., 0]).all() and np.isnan(cent[..., 1:]).all()
        else:
            assert np.isposinf(cent[:, 0]).all() and (cent[:, 1:] == 0).all()
    g.close()


@pytest.mark.parametrize("rows", [128, 129])  # 48,896 / 49,278 seeds a side
def test_many_seeds_and_clusters_gpu(gpu, rows):
    """32 clusters: the k-means is the device's up to 49,152 seeds a side, the
    host's above."""
    shape = (382, 400, 1)
    say("case widget many seeds and clusters", rows)
    rgba, fg, bg = random_case(shape, rows)
    fg, bg = np.zeros((400, 382), np.uint8), np.zeros((400, 382), np.uint8)
    fg[:rows] = 1
    bg[400 - rows:] = 1
    check(gpu, shape, rgba, fg.ravel(), bg.ravel(), dict(lazy=True, k=32, kmeans_iterations=4),
          solve=False)
