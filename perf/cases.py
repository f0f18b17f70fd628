"""Workloads of the grid-cut library, as programs call it.

Each case is one kind of program over one grid:

  segment   interactive segmentation: data term from an image and seeds in
            HBM, cut, flow and labels
  resolve   a cut whose capacities another kernel wrote in place
            (input_planes / inputs_written), flow and labels
  widget    the reference widget's "Model" and "Cut" buttons: its own data
            terms, cut, labels, tag post-process
  hostgraph a graph that arrives in host memory (a loaded graph file): folded
            terminal capacities and arcs set from numpy, labels back in numpy
  train     the differentiable cut: energy and the gradients of every capacity
  batch     uneven instances in one graph: cut all, gradients of all

listed() holds the sizes and options of this repository's own configurations
(jfcut.CONFIGS, the reference's fixtures, the batched configuration) and
generic small, odd and ordinary ones; draw() spreads over the same ranges.
Images, seeds and graphs come from the library's generators or from a seeded
torch generator; every result is a whole number.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "jf-cut_amd"))
import jfcut  # noqa: E402

_SEGMENT = dict(kind="segment", nz=1, data="rgb8", lam=50.0, k=5, unary=100, tags=False,
                tile_shape="default", max_local_iters=0, initial_relabel=-1, stall_certify=-1)
_WIDGET = dict(kind="widget", nz=1, lazy=True, k=8, iterations=32)


def listed():
    return [
        # a training step on a small patch: launch latency and host work
        dict(name="train_patch_96x80_4c", kind="train", nx=96, ny=80, conn=4),
        # a training step on an image, odd rows, diagonals
        dict(name="train_1023x767_8c", kind="train", nx=1023, ny=767, conn=8),
        # one stroke of interactive segmentation on a preview
        dict(_SEGMENT, name="segment_512x512_4c", nx=512, ny=512, conn=4),
        # the reference widget on an image of its fixtures' size
        dict(_WIDGET, name="widget_600x450_4c", nx=600, ny=450, conn=4),
        # a loaded graph file of the reference's fixture size
        dict(name="hostgraph_640x480_4c", kind="hostgraph", nx=640, ny=480, nz=1, conn=4),
        # a 12-megapixel photograph
        dict(_SEGMENT, name="segment_4000x3000_8c", nx=4000, ny=3000, conn=8),
        # strokes alone decide (no unary term): flow crosses the whole image
        dict(_SEGMENT, name="strokes_3750x2500_8c", nx=3750, ny=2500, conn=8, unary=0),
        # the large 2D cut of the benchmark, capacities written in place, under
        # the settings its autotuner keeps
        dict(_SEGMENT, name="resolve_15000x10000_8c", kind="resolve", nx=15000, ny=10000, conn=8,
             max_local_iters=2, initial_relabel=0, stall_certify=1),
        # the video volume of the benchmark, under its tuned settings
        dict(_SEGMENT, name="video_2560x1440x50_6c", nx=2560, ny=1440, nz=50, conn=6,
             data="video", tile_shape="32x4x2", max_local_iters=2, initial_relabel=1,
             stall_certify=1),
        # the 16-bit scan of the benchmark, under its tuned settings
        dict(_SEGMENT, name="volume_512x512x512_6c", nx=512, ny=512, nz=512, conn=6,
             data="u16", lam=40.0, k=4, max_local_iters=4),
        # a brain-atlas sized scan, every side odd, with the tag post-process
        dict(_SEGMENT, name="scan_181x217x181_6c", nx=181, ny=217, nz=181, conn=6,
             data="u16", lam=40.0, k=4, tags=True),
        # the batched configuration: 256 uneven images, forward and backward
        dict(name="batch_256_mixed", kind="batch", count=256, first=0),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["segment2d", "segment2d", "segment3d", "widget", "hostgraph", "train",
                       "batch", "resolve"])
    lam = round(rng.uniform(20.0, 80.0), 1)
    if kind == "segment2d":
        unary = rng.choice([100, 100, 100, 0])
        nx = log(64, 1600 if unary == 0 else 6000)
        return dict(_SEGMENT, nx=nx, ny=max(32, int(nx * rng.uniform(0.5, 1.5))),
                    conn=rng.choice([4, 8]), data=rng.choice(["rgb8", "rgb8", "u8", "u16"]),
                    lam=lam, k=rng.randint(2, 8), unary=unary, tags=rng.random() < 0.3,
                    tile_shape=rng.choice(["default", "default", "64x4", "16x16"]),
                    initial_relabel=rng.choice([-1, 0, 1]), stall_certify=rng.choice([-1, 0, 1]))
    if kind == "segment3d":
        data = rng.choice(["video", "u16"])
        nx = log(40, 512)
        return dict(_SEGMENT, nx=nx, ny=max(32, int(nx * rng.uniform(0.5, 1.5))),
                    nz=rng.randint(8, 100), conn=6, data=data, lam=lam, k=rng.randint(2, 6),
                    tags=rng.random() < 0.3, tile_shape=rng.choice(["default", "32x4x2"]),
                    max_local_iters=rng.choice([0, 2, 4]), initial_relabel=rng.choice([-1, 1]))
    if kind == "widget":
        nx = log(64, 2000)
        nz = rng.choice([1, 1, rng.randint(4, 24)])
        nx = min(nx, 400) if nz > 1 else nx
        return dict(_WIDGET, nx=nx, ny=max(32, int(nx * rng.uniform(0.5, 1.5))), nz=nz,
                    conn=6 if nz > 1 else 4, lazy=rng.random() < 0.6, k=rng.randint(2, 16))
    if kind == "hostgraph":
        nx = log(64, 1500)
        return dict(kind="hostgraph", nx=nx, ny=max(32, int(nx * rng.uniform(0.5, 1.5))), nz=1,
                    conn=rng.choice([4, 8]))
    if kind == "train":
        nx = log(24, 2000)
        return dict(kind="train", nx=nx, ny=max(16, int(nx * rng.uniform(0.5, 1.5))),
                    conn=rng.choice([4, 8]))
    if kind == "batch":
        return dict(kind="batch", count=log(2, 200), first=rng.randrange(1, 1 << 20))
    nx = log(200, 10000)
    return dict(_SEGMENT, kind="resolve", nx=nx, ny=max(64, int(nx * rng.uniform(0.4, 1.0))),
                conn=rng.choice([4, 8]), lam=lam, max_local_iters=rng.choice([0, 2, 3, 4]),
                initial_relabel=rng.choice([-1, 0, 1]), stall_certify=rng.choice([-1, 0, 1]))


# ---- inputs ---------------------------------------------------------------------


def _image(c, seed):
    """(image, seed map) of a segment / resolve case, on the GPU."""
    if c["data"] == "video":
        img, sd = jfcut.synth_video(c["nx"], c["ny"], c["nz"], seed=seed)
    elif c["data"] == "u16" and c["nz"] > 1:
        img, sd = jfcut.synth_volume(c["nx"], c["ny"], c["nz"], seed=seed)
    else:
        img, sd = jfcut.synth_image(c["nx"], c["ny"],
                                    nblobs=40 if c["nx"] * c["ny"] > 1 << 22 else 8, seed=seed)
        if c["data"] != "rgb8":  # grey, 8 or 16 bits
            img = np.ascontiguousarray(img[..., 0])
            if c["data"] == "u16":
                img = img.astype(np.uint16) * 257
    # torch kernels do not take uint16; the library reads the 16-bit words
    if img.dtype == np.uint16:
        img = img.view(np.int16)
    return torch.from_numpy(img).cuda(), torch.from_numpy(sd).cuda()


def _model(c, g, img, sd):
    rng = 65535 if c["data"] == "u16" and c["nz"] == 1 else 1024 if c["data"] == "u16" else 255
    video = c["data"] == "video"
    g.model_image(img, sd, k_fg=c["k"], k_bg=c["k"], unary_scale=c["unary"], rng=rng,
                  lambda_xy=c["lam"], lambda_z=0.6 * c["lam"] if video else c["lam"],
                  z_separate=1 if video else 0)


def _options(c):
    return dict(tile_shape=c["tile_shape"], max_local_iters=c["max_local_iters"],
                initial_relabel=c["initial_relabel"], stall_certify=c["stall_certify"])


# direction d -> (dy, dx): +x -x +y -y (+x+y) (-x-y) (-x+y) (+x-y)
_OFF = [(0, 1), (0, -1), (1, 0), (-1, 0), (1, 1), (-1, -1), (1, -1), (-1, 1)]


def _shift(a, dy, dx, fill):
    """b[y, x] = a[y + dy, x + dx], `fill` outside the grid."""
    b = np.full_like(a, fill)
    h, w = a.shape
    b[max(0, -dy):h - max(0, dy), max(0, -dx):w - max(0, dx)] = \
        a[max(0, dy):h - max(0, -dy), max(0, dx):w - max(0, -dx)]
    return b


def _capacities(nx, ny, conn, seed):
    """A trained unary over a noisy object and contrast-weighted arcs: whole
    numbers cs, ct (ny, nx) and caps (conn, ny, nx)."""
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:ny, 0:nx]
    cy, cx = ny * rng.uniform(0.4, 0.6), nx * rng.uniform(0.4, 0.6)
    inside = ((y - cy) / (0.3 * ny)) ** 2 + ((x - cx) / (0.35 * nx)) ** 2 < 1
    grey = np.where(inside, 170.0, 90.0) + rng.normal(0, 30, (ny, nx))
    logit = (grey - 130.0) * 0.8
    cs = np.maximum(np.rint(logit), 0).astype(np.int32)
    ct = np.maximum(np.rint(-logit), 0).astype(np.int32)
    caps = np.zeros((conn, ny, nx), np.int32)
    for d in range(conn):
        dy, dx = _OFF[d]
        diff = _shift(grey, dy, dx, np.inf) - grey
        lam = 50.0 if d < 4 else 50.0 / math.sqrt(2.0)
        caps[d] = np.rint(lam * np.exp(-diff * diff / (2.0 * 45.0 ** 2))).astype(np.int32)
    return cs, ct, caps


def prepare(case, seed):
    c, kind = case, case["kind"]
    st = {"case": c}
    if kind in ("segment", "resolve"):
        n = c["nx"] * c["ny"] * c["nz"]
        img, sd = _image(c, seed)
        g = jfcut.GridGraph.grid(c["nx"], c["ny"], c["nz"], c["conn"])
        st.update(g=g, opt=_options(c), labels=torch.empty(n, dtype=torch.uint8, device="cuda"))
        if kind == "segment":
            st.update(img=img, sd=sd)
            if c["tags"]:
                st.update(fg=(sd.reshape(-1) == 1).to(torch.uint8),
                          tags=torch.empty(n, dtype=torch.uint8, device="cuda"))
        else:
            _model(c, g, img, sd)
    elif kind == "widget":
        if c["nz"] > 1:
            img, sd = jfcut.synth_video(c["nx"], c["ny"], c["nz"], seed=seed)
        else:
            img, sd = jfcut.synth_image(c["nx"], c["ny"], seed=seed)
        n = sd.size
        rgba = np.full((n, 4), 255, np.uint8)
        rgba[:, :3] = img.reshape(n, 3)
        sd = torch.from_numpy(sd.reshape(-1)).cuda()
        st.update(g=jfcut.GridGraph.grid(c["nx"], c["ny"], c["nz"], c["conn"]),
                  rgba=torch.from_numpy(rgba).cuda(), fg=(sd == 1).to(torch.uint8),
                  bg=(sd == 2).to(torch.uint8),
                  labels=torch.empty(n, dtype=torch.uint8, device="cuda"),
                  tags=torch.empty(n, dtype=torch.uint8, device="cuda"))
    elif kind == "hostgraph":
        cs, ct, caps = _capacities(c["nx"], c["ny"], c["conn"], seed)
        st.update(g=jfcut.GridGraph.grid(c["nx"], c["ny"], c["nz"], c["conn"]), ef=cs - ct,
                  caps=caps)
    elif kind == "train":
        cs, ct, caps = _capacities(c["nx"], c["ny"], c["conn"], seed)
        st.update(
            cs=torch.from_numpy(cs.reshape(-1)).cuda().float().requires_grad_(),
            ct=torch.from_numpy(ct.reshape(-1)).cuda().float().requires_grad_(),
            w=torch.from_numpy(caps.reshape(c["conn"], -1)).cuda().float().requires_grad_())
    else:  # batch
        specs = jfcut.batch_specs(c["count"], seed=c["first"])
        g = jfcut.GridGraph([(s["W"], s["H"], 1, s["conn"]) for s in specs])
        for i, s in enumerate(specs):
            img, sd = jfcut.synth_image(s["W"], s["H"], seed=1000 * seed + i)
            g.model_image(img, sd, inst=i, lambda_xy=s["lam"])
        n, k = g.size()
        st.update(g=g, grads=(torch.zeros(n, device="cuda"), torch.zeros(n, device="cuda"),
                              torch.zeros(k, n, device="cuda")))
    return st


def run(state):
    c, kind = state["case"], state["case"]["kind"]
    if kind == "train":
        cs, ct, w = state["cs"], state["ct"], state["w"]
        energy = jfcut.min_cut_energy(cs, ct, w, (c["nx"], c["ny"], 1), c["conn"])
        return (energy.detach(),) + torch.autograd.grad(energy, (cs, ct, w))
    g = state["g"]
    if kind == "segment":
        _model(c, g, state["img"], state["sd"])
        g.solve(**state["opt"])
        out = {"flow": g.flow(), "labels": g.labels(out=state["labels"])}
        if c["tags"]:
            out["tags"] = g.tags(state["fg"], out=state["tags"])
        return out
    if kind == "resolve":
        g.inputs_written()
        g.solve(**state["opt"])
        return {"flow": g.flow(), "labels": g.labels(out=state["labels"])}
    if kind == "widget":
        g.model_widget(state["rgba"], state["fg"], state["bg"], lazy=c["lazy"], k=c["k"],
                       kmeans_iterations=c["iterations"])
        g.solve()
        return {"flow": g.flow(), "labels": g.labels(out=state["labels"]),
                "tags": g.tags(state["fg"], out=state["tags"])}
    if kind == "hostgraph":
        g.set_excess(state["ef"])
        g.set_all_neighbor_caps(state["caps"])
        g.solve()
        return {"flow": g.flow(), "labels": g.labels()}
    for i in range(len(g.shapes)):
        g.inputs_written(i)
    g.solve()
    return (g.flows(),) + tuple(g.backward_all(out=state["grads"]))


def work(case):
    """Inputs read once, outputs written once; one compare or add per input
    capacity or pixel word."""
    c, kind = case, case["kind"]
    if kind == "batch":
        b = f = 0
        for s in jfcut.batch_specs(c["count"], seed=c["first"]):
            n = s["W"] * s["H"]
            b += n * (4 * (2 + s["conn"]) + 4 * (2 + s["conn"]))
            f += n * (2 + s["conn"])
        return {"bytes": b, "flops": f}
    n = c["nx"] * c["ny"] * c.get("nz", 1)
    if kind == "segment":
        px = {"rgb8": 3, "video": 3, "u8": 1, "u16": 2}[c["data"]]
        return {"bytes": n * (px + 2 + (2 if c["tags"] else 0)), "flops": n * (2 + c["conn"])}
    if kind == "widget":
        return {"bytes": n * (4 + 2 + 2), "flops": n * (2 + c["conn"])}
    if kind == "train":  # float capacities in, float gradients out
        return {"bytes": n * 8 * (2 + c["conn"]), "flops": n * (2 + c["conn"])}
    terms = 1 if kind == "hostgraph" else 2
    return {"bytes": n * (4 * (terms + c["conn"]) + 1), "flops": n * (2 + c["conn"])}


# ---- exact results of small training steps ------------------------------------------


def _min_cut(cs, ct, caps):
    """(flow, minimal source side) by push-relabel over whole-grid arrays."""
    k = len(caps)
    e = cs.astype(np.int64) - ct
    r = caps.astype(np.int64).copy()
    inf = e.size + 1

    def distances():
        h = np.where(e < 0, 0, inf)
        while True:
            n = h
            for d in range(k):
                n = np.where(r[d] > 0, np.minimum(n, _shift(h, *_OFF[d], inf) + 1), n)
            if (n == h).all():
                return h
            h = n

    h = distances()
    step = 0
    while ((e > 0) & (h < inf)).any():
        for d in range(k):
            dy, dx = _OFF[d]
            f = np.where((e > 0) & (h < inf) & (h == _shift(h, dy, dx, inf) + 1),
                         np.minimum(e, r[d]), 0)
            back = _shift(f, -dy, -dx, 0)
            e += back - f
            r[d] -= f
            r[d ^ 1] += back
        m = np.full_like(h, inf)
        for d in range(k):
            m = np.where(r[d] > 0, np.minimum(m, _shift(h, *_OFF[d], inf) + 1), m)
        h = np.where((e > 0) & (m > h), m, h)
        step += 1
        if step % 40 == 0:
            h = distances()
    flow = int(np.minimum(cs, ct).sum() + np.maximum(ct - cs, 0).sum() - np.maximum(-e, 0).sum())
    s = e > 0
    while True:
        n = s
        for d in range(k):
            dy, dx = _OFF[d]
            n = n | _shift(s & (r[d] > 0), -dy, -dx, False)
        if (n == s).all():
            return flow, s
        s = n


def exact(case, seed):
    """Energy and gradients of a small training step; other cases return whole
    numbers of solves too large for a plain array program."""
    c = case
    if c["kind"] != "train" or c["nx"] * c["ny"] > 40000:
        return None
    cs, ct, caps = _capacities(c["nx"], c["ny"], c["conn"], seed)
    flow, s = _min_cut(cs.astype(np.int64), ct.astype(np.int64), caps)
    dw = np.stack([s & ~_shift(s, *_OFF[d], True) for d in range(c["conn"])])
    return (np.float64(flow), (~s).astype(np.float64).reshape(-1),
            s.astype(np.float64).reshape(-1), dw.astype(np.float64).reshape(c["conn"], -1))
