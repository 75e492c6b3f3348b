"""The row-run sampler where its lists and its LDS fill up, against the oracle
bit for bit.  One wave per ray: more than 1024 candidates within the bound, in
buckets below the 48-hit cap, on surfaces deep behind each other (the list stops
32 slots behind the first hit) and where the walk has to go on behind that.
Tiles: windows of more than eight columns, buffers of 16, rows of more points
than the LDS holds, with and without deferral.  Each scene's precondition is
checked on the host."""
import numpy as np
import pytest
import torch

import epcq.csrc as C
import test_gpu_rows
from epcq import synth
from epcq.epcq import RenderOptions
from scenes import bits, to_dev
from test_gpu_sampling import View, check_dense, compact_vs_dense
from test_gpu_wave import heavy_threshold

pytestmark = pytest.mark.gpu

LIST = 1024  # positions that a wave's list holds
LDS_ROW = 960  # points of a window row that a tile stages at once
BUCKET = 48  # hits that a bucket gives


def camera(W, H):
    return synth.look_at_camera([2.2, -2.4, 2.1], W, H, 1.39 * max(W, 48))


def unproject(cam, u, v, z):
    """Points at depth z before the pixels (u, v) (both with their jitter)."""
    p = np.stack([(u - cam.cx) / cam.fx * z, (v - cam.cy) / cam.fy * z, z], axis=-1)
    return (p @ np.asarray(cam.c2w)[:3, :3].T + np.asarray(cam.c2w)[:3, 3]).astype(np.float32)


def volume(cam, per_pixel, near, far, rng):
    """per_pixel points before every pixel, at depths spread over [near, far]."""
    u, v = np.meshgrid(np.arange(cam.width), np.arange(cam.height))
    u, v = np.repeat(u.ravel(), per_pixel), np.repeat(v.ravel(), per_pixel)
    jitter = lambda: rng.uniform(0.3, 0.7, u.size)  # noqa: E731
    pts = unproject(cam, u + jitter(), v + jitter(), rng.uniform(near, far, u.size))
    return np.ascontiguousarray(pts[rng.permutation(len(pts))])


def near_the_ray(v, u, vv, r):
    """Points of the window of pixel (u, vv) within r of the line through it."""
    k = v.opt.kernel_size
    ko = (k + 1) // 2
    ids = []
    for y in range(vv + 1 - ko, vv + 1 - ko + k):
        for x in range(u + 1 - ko, u + 1 - ko + k):
            s, n = v.oh.reshape(v.cam.height, v.cam.width, 2)[y, x]
            if n > 0:
                ids.append(v.oi[s:s + n])
    p = v.pts[np.concatenate(ids)].astype(np.float64)
    o = np.asarray(v.cam.c2w, np.float64)[:3, 3]
    d = unproject(v.cam, np.float64(u), np.float64(vv), np.float64(1.0)) - o
    d /= np.linalg.norm(d)
    w = p - o
    return int((np.linalg.norm(w - (w @ d)[:, None] * d, axis=1) < (r if np.ndim(r) == 0 else r[np.concatenate(ids)])).sum())


# options, depths of the points
WAVE = {
    # the list is cut and the walk ends in it
    "deep": (dict(), (2.0, 6.0)),
    "deep-one-sample": (dict(num_sample_points_per_ray=1), (2.0, 6.0)),
    # a walk that emits nothing or too little within the list goes on
    "faint": (dict(sdf2weight_gaussian_gamma=0.0005), (2.0, 6.0)),
    "thin-slots": (dict(t_intvl=1e-5), (2.0, 6.0)),
    "few-slots": (dict(t_intvl=3e-4), (2.0, 6.0)),
    # too many even within the list's depth
    "shallow": (dict(), (2.0, 2.2)),
    "no-depth": (dict(t_intvl=0.0), (2.0, 6.0)),
}


@pytest.mark.parametrize("k,K,mode", [(9, 8, "knn"), (9, 8, "compat"), (12, 16, "knn"), (16, 32, "knn")])
@pytest.mark.parametrize("what", list(WAVE))
def test_wave_lists(dev, what, k, K, mode):
    opts, (near, far) = WAVE[what]
    W, H = 44, 34
    cam = camera(W, H)
    rng = np.random.default_rng(k)
    pts = volume(cam, 34 if k == 9 else 22, near, far, rng)
    r = 0.3
    v = View(pts, cam, dev, **dict(dict(kernel_size=k, radius_threshold=r, num_point_cloud_per_sp=K,
                                        num_sample_points_per_ray=2), **opts))
    assert C.sampling_form(v.opt, len(pts), H, W) == C.FORM_ROW_WAVES
    assert v.oh[:, 1].max() <= BUCKET
    assert min(near_the_ray(v, u, y, r) for u, y in ((22, 17), (15, 12), (30, 20))) > LIST
    print("wave list", what, k, K, mode, len(pts), flush=True)
    check_dense(v, mode)
    compact_vs_dense(v, mode)
    rays = rng.integers(0, W * H, 15 * W * H // k**2).astype(np.int32)
    if k <= 12:
        assert C.sampling_form(v.opt, len(pts), H, W, rays=len(rays)) == C.FORM_ROW_WAVES
    compact_vs_dense(v, mode, rays=rays)              # with the copy and its bounds (k <= 12)
    compact_vs_dense(v, mode, rays=rays, cull=False)  # the bounds worked out on the way
    compact_vs_dense(v, mode, rays=rays[:3])          # a list too short for the copy


def test_wave_lists_per_point_radius(dev):
    W, H = 44, 34
    cam = camera(W, H)
    rng = np.random.default_rng(5)
    pts = volume(cam, 34, 2.0, 6.0, rng)
    radius = rng.uniform(0.28, 0.4, len(pts)).astype(np.float32)
    v = View(pts, cam, dev, radius=radius, kernel_size=9, radius_threshold=0.4, num_point_cloud_per_sp=16,
             num_sample_points_per_ray=2)
    assert v.oh[:, 1].max() <= BUCKET and near_the_ray(v, 22, 17, radius) > LIST
    feat = torch.randn(len(pts), 12, generator=torch.Generator().manual_seed(3)).to(dev)
    print("wave list, per-point radius", flush=True)
    compact_vs_dense(v, "knn", feat=feat)
    compact_vs_dense(v, "knn", rays=rng.integers(0, W * H, 600).astype(np.int32), feat=feat, cull=False)


@pytest.mark.parametrize("hot,per_pixel,k,K,mode,opts", [
    # buckets beyond the 48-hit cap, and more candidates within the bound than the list holds
    (0, 70, 5, 8, "knn", dict()),
    (0, 70, 9, 16, "knn", dict(num_sample_points_per_ray=1)),
    (0, 70, 9, 8, "compat", dict(sdf2weight_gaussian_gamma=0.0005)),
    (0, 130, 7, 32, "knn", dict(t_intvl=3e-4)),
    # a bucket of more chunks than the list holds, beside ordinary ones
    (90_000, 20, 5, 8, "knn", dict()),
    (90_000, 20, 5, 8, "compat", dict()),
    (90_000, 60, 9, 16, "knn", dict()),
    # and one whose chunks it holds
    (20_000, 20, 9, 8, "knn", dict()),
    (20_000, 60, 3, 8, "compat", dict()),
])
def test_wave_full_buckets(dev, hot, per_pixel, k, K, mode, opts):
    W, H = 44, 34
    cam = camera(W, H)
    rng = np.random.default_rng(hot + k)
    pts = volume(cam, per_pixel, 3.0, 3.6, rng)
    if hot:  # before one pixel, on two surfaces
        z = rng.choice([3.0, 3.2], hot) + rng.normal(0, 0.01, hot)
        pts = np.concatenate([pts, unproject(cam, 22 + rng.uniform(0.3, 0.7, hot), 17 + rng.uniform(0.3, 0.7, hot), z)])
        pts = np.ascontiguousarray(pts[rng.permutation(len(pts))])
    r = 0.2
    v = View(pts, cam, dev, **dict(dict(kernel_size=k, radius_threshold=r, num_point_cloud_per_sp=K,
                                        num_sample_points_per_ray=2), **opts))
    assert C.sampling_form(v.opt, len(pts), H, W) == C.FORM_ROW_WAVES
    most = v.oh[:, 1].max()
    assert most > BUCKET and near_the_ray(v, 22, 17, r) > LIST
    assert (most > 64 * LIST) == (hot == 90_000)
    print("wave full buckets", hot, per_pixel, k, K, mode, flush=True)
    check_dense(v, mode)
    compact_vs_dense(v, mode)
    rays = np.concatenate([rng.integers(0, W * H, 250), [17 * W + 22]]).astype(np.int32)
    assert C.sampling_form(v.opt, len(pts), H, W, rays=len(rays)) == C.FORM_ROW_WAVES
    feat = torch.randn(len(pts), 9, generator=torch.Generator().manual_seed(3)).to(dev)
    compact_vs_dense(v, mode, rays=rays)
    compact_vs_dense(v, mode, rays=rays, cull=False)
    compact_vs_dense(v, mode, rays=rays, feat=feat)


def patched(cam, n, per_pixel, x0, y0, w, h, rng):
    """n points over the whole image and per_pixel before each pixel of a patch."""
    u, y = np.meshgrid(np.arange(x0, x0 + w), np.arange(y0, y0 + h))
    u, y = np.repeat(u.ravel(), per_pixel), np.repeat(y.ravel(), per_pixel)
    u = np.concatenate([u + rng.uniform(0.3, 0.7, u.size), rng.uniform(0, cam.width, n)])
    y = np.concatenate([y + rng.uniform(0.3, 0.7, y.size), rng.uniform(0, cam.height, n)])
    # a surface with some relief, so that most pixels have hits close together
    z = 3.0 + 0.2 * np.sin(u / 9.0) * np.cos(y / 7.0) + rng.normal(0, 0.003, u.size)
    pts = unproject(cam, u, y, z)
    return np.ascontiguousarray(pts[rng.permutation(len(pts))])


TILES = [
    # W, H, k, K, mode, points over the image, points per pixel and patch, features, per-point radius, S
    (640, 420, 16, 16, "knn", 40_000, 0, (0, 0, 0, 0), 32, True),
    (640, 420, 16, 16, "compat", 40_000, 0, (0, 0, 0, 0), 7, False),
    (650, 410, 11, 9, "knn", 60_000, 0, (0, 0, 0, 0), 5, False),
    (650, 410, 9, 16, "compat", 80_000, 0, (0, 0, 0, 0), 0, True),
    (650, 410, 12, 12, "knn", 60_000, 0, (0, 0, 0, 0), 0, False),
    # a region's rows of 961 .. 3840 points
    (650, 410, 9, 16, "knn", 40_000, 20, (170, 120, 70, 20), 16, False),
    (650, 410, 9, 8, "compat", 40_000, 30, (170, 120, 90, 20), 0, False),
    (650, 410, 10, 16, "knn", 40_000, 20, (170, 120, 70, 20), 4, True),
    # and at the image's corner, where clamping repeats them
    (650, 410, 9, 8, "knn", 40_000, 20, (0, 0, 70, 20), 0, False),
    # rows too long for windows of up to eight columns
    (430, 310, 8, 8, "knn", 40_000, 20, (170, 120, 70, 20), 0, False),
]


@pytest.mark.parametrize("heavy", [C.HEAVY_DEFAULT, 0, 1])
@pytest.mark.parametrize("case", TILES, ids=lambda c: f"{c[0]}x{c[1]}-k{c[2]}-K{c[3]}-{c[4]}-{c[6]}-F{c[8]}")
def test_tiles(dev, case, heavy):
    W, H, k, K, mode, n, per_pixel, patch, F, per_point = case
    cam = camera(W, H)
    rng = np.random.default_rng(W + k)
    pts = patched(cam, n, per_pixel, *patch, rng) if per_pixel else patched(cam, n, 1, 0, 0, 1, 1, rng)
    radius = (0.02 * np.exp(-1.2 * rng.random(len(pts)))).astype(np.float32) if per_point else None
    v = View(pts, cam, dev, radius=radius, kernel_size=k, radius_threshold=0.02, num_point_cloud_per_sp=K,
             num_sample_points_per_ray=2)
    rows = v.oh[:, 1].reshape(H, W)
    if per_pixel:
        # the widest run of the 64 + k - 1 columns of a tile, over all tiles
        ko = (k + 1) // 2
        longest = max(rows[:, max(0, u0 - ko + 1):u0 + 64 + k - ko].clip(0).sum(1).max() for u0 in range(0, W, 64))
        assert LDS_ROW < longest < 4 * LDS_ROW
    with heavy_threshold(heavy):
        assert C.sampling_form(v.opt, len(pts), H, W) == C.FORM_ROW_TILES
        feat = None
        if F:
            feat = torch.randn(len(pts), F, generator=torch.Generator().manual_seed(2)).to(dev)
            feat = feat.to(torch.bfloat16) if F > 16 else feat
        print("tiles", case, heavy, flush=True)
        out = compact_vs_dense(v, mode, feat=feat)
        assert int((out["n_samples"] > 0).sum()) > 3000
        if C.sampling_form(v.opt, len(pts), H, W, compact=False) == C.FORM_ROW_TILES:
            check_dense(v, mode)


@pytest.mark.parametrize("case", [
    ("thin", 515, 513, dict(radius_threshold=0.02, kernel_size=9), "compat", False, None),
    ("thin", 515, 513, dict(t_intvl=0.0003, radius_threshold=0.02, kernel_size=9), "knn", False, None),
    ("box", 570, 461, dict(kernel_size=16, num_point_cloud_per_sp=16), "knn", True, (torch.bfloat16, 32)),
    ("box", 4, 65537, dict(kernel_size=15), "compat", False, (torch.float32, 4)),
    ("hot", 513, 515, dict(kernel_size=9), "knn", False, None),
    # windows of one and two columns, on an image of few tiles
    ("dense", 260, 200, dict(kernel_size=1), "knn", True, None),
    ("dense", 261, 203, dict(kernel_size=1), "compat", False, (torch.float32, 5)),
    ("dense", 366, 359, dict(kernel_size=2), "knn", True, None),
    ("far", 380, 260, dict(radius_threshold=0.01, kernel_size=8), "knn", False, None),
], ids=lambda c: f"{c[0]}-{c[1]}x{c[2]}-{c[4]}-k{c[3]['kernel_size']}")
def test_tiles_by_window(dev, case):
    kind, W, H, opts, _, per_point, _ = case
    pts, _ = test_gpu_rows.scene(kind, W, H)
    assert C.sampling_form(RenderOptions(**opts), len(pts), H, W, live=2 if per_point else None) == C.FORM_ROW_TILES
    test_gpu_rows.test_rows_equal_lane_sets(dev, case)


@pytest.mark.parametrize("W,H,n,form", [(200, 150, 60_000, C.FORM_ROW_WAVES), (430, 310, 120_000, C.FORM_ROW_TILES)])
def test_captured_and_on_two_streams(dev, W, H, n, form):
    """The calls inside a captured graph, replayed between other work, and two
    images at once on two streams, each with its own workspace and queue."""
    cam = camera(W, H)
    rng = np.random.default_rng(9)
    v = View(patched(cam, n, 30, 20, 20, 90, 20, rng), cam, dev, kernel_size=5, radius_threshold=0.02,
             num_point_cloud_per_sp=8)
    total = len(v.pts)
    assert C.sampling_form(v.opt, total, H, W) == form
    feat = torch.randn(total, 8, generator=torch.Generator().manual_seed(2)).to(dev)
    rays = to_dev(rng.integers(0, W * H, 2000).astype(np.int32), dev)

    def calls():
        idx, _, table = v.npts.pts2plane(v.cs, v.opt)
        return [v.npts.knn_sampling(v.cs, v.opt, idx, table, feat=feat),
                v.npts.knn_sampling(v.cs, v.opt, idx, table, rays=rays),
                dict(zip("xitm", v.npts.render_image_hashtable_topk(v.cs, v.opt, idx, None, table)))]

    def equal(a, b):
        for x, y in zip(a, b):
            for key in x:
                assert np.array_equal(bits(x[key].cpu().numpy()), bits(y[key].cpu().numpy())), key

    print("capture", W, H, flush=True)
    want = calls()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        calls()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = calls()
    for i in range(3):
        for d in got:
            for t in d.values():
                t.view(torch.uint8).fill_(0x5A)
        graph.replay()
        torch.cuda.synchronize()
        equal(got, want)
        calls()
    print("two streams", W, H, flush=True)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [[], []]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    for _ in range(4):
        for s, o in zip(streams, outs):
            with torch.cuda.stream(s):
                o.append(calls())
    torch.cuda.synchronize()
    for o in outs:
        for x in o:
            equal(x, want)
