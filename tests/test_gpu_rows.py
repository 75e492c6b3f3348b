"""The row-run sampler (full images and short ray lists) against the lane-set
sampler, which a call without a workspace takes (cull=False): every output
bit for bit, at the edges of its tiles, windows and rules, and against the
oracle on a few."""
import numpy as np
import pytest
import torch

from epcq import synth
from epcq.epcq import NeuralPoints, RenderOptions
from oracle import oracle
from scenes import bits, camera_spec, to_dev

pytestmark = pytest.mark.gpu


def scene(kind, W, H, seed=0):
    rng = np.random.default_rng(seed)
    cam = synth.look_at_camera([2.2, -2.4, 2.1], W, H, 1.39 * max(W, 48))
    if kind == "box":
        pts = synth.box_scene(60_000, n_boxes=12, seed=seed)
    elif kind == "dense":  # several points per pixel, buckets beyond the 48-hit cap
        pts = synth.box_scene(400_000, n_boxes=6, seed=seed)
    elif kind == "hot":  # a pixel with most of the points
        pts = np.concatenate([synth.sphere_cloud(5_000, seed=seed),
                              np.repeat(np.float32([[0.01, 0.02, 0.03]]), 30_000, axis=0)
                              + rng.normal(0, 1e-4, (30_000, 3)).astype(np.float32)])
    elif kind == "thin":  # single hits before surfaces
        pts = np.concatenate([rng.uniform(-1, 1, (4_000, 3)).astype(np.float32), synth.sphere_cloud(30_000, seed=seed)])
    elif kind == "inside":  # points around and behind the camera
        pts = rng.uniform(-3, 3, (50_000, 3)).astype(np.float32)
        cam = synth.look_at_camera([0.3, -0.2, 0.1], W, H, 0.5 * max(W, 48))
    else:
        assert kind == "far"  # a large origin
        pts = synth.box_scene(30_000, n_boxes=12, seed=seed) + np.float32([800, -500, 300])
        cam.c2w[:, 3] += np.float32([800, -500, 300])
        cam.w2c[:, 3] -= cam.w2c[:, :3] @ np.float32([800, -500, 300])
    return np.ascontiguousarray(pts, np.float32), cam


CASES = [
    # kind, W, H, options, mode, per-point radius, feature dtype and width
    ("box", 1, 1, dict(), "compat", False, None),
    ("box", 63, 5, dict(), "knn", False, (torch.float32, 5)),
    ("box", 64, 4, dict(kernel_size=1), "compat", True, None),
    ("box", 65, 3, dict(kernel_size=2, num_point_cloud_per_sp=3), "knn", False, None),
    ("box", 130, 9, dict(kernel_size=16, num_point_cloud_per_sp=16), "knn", True, (torch.bfloat16, 32)),
    ("box", 129, 66, dict(kernel_size=8, num_point_cloud_per_sp=32), "knn", True, (torch.bfloat16, 7)),
    ("box", 2, 40, dict(kernel_size=15), "compat", False, (torch.float32, 4)),
    ("dense", 70, 50, dict(), "compat", False, None),
    ("dense", 130, 40, dict(kernel_size=7), "knn", True, None),
    ("dense", 48, 36, dict(kernel_size=11, num_point_cloud_per_sp=9), "knn", False, (torch.float32, 16)),
    ("hot", 96, 64, dict(), "compat", False, None),
    ("hot", 96, 64, dict(kernel_size=9), "knn", False, None),
    ("thin", 100, 75, dict(radius_threshold=0.02), "compat", False, None),
    ("thin", 100, 75, dict(t_intvl=0.0003, radius_threshold=0.02), "knn", False, None),
    ("thin", 100, 75, dict(t_intvl=-0.01), "compat", False, None),
    ("thin", 100, 75, dict(t_intvl=0.0), "compat", False, None),
    ("inside", 90, 60, dict(radius_threshold=0.05), "knn", False, None),
    ("inside", 90, 60, dict(radius_threshold=1.5, kernel_size=3), "compat", False, None),
    ("far", 80, 60, dict(radius_threshold=0.01), "knn", False, None),
    ("box", 80, 60, dict(radius_threshold=float("inf")), "compat", False, None),
    ("box", 80, 60, dict(radius_threshold=0.0), "knn", False, None),
    ("box", 80, 60, dict(num_sample_points_per_ray=1), "compat", False, None),
    # images large enough for the tiles of 64 x 4 rays
    ("box", 363, 363, dict(), "compat", False, None),
    ("box", 385, 341, dict(kernel_size=8, num_point_cloud_per_sp=32), "knn", True, (torch.bfloat16, 7)),
    ("box", 400, 330, dict(kernel_size=16, num_point_cloud_per_sp=16), "knn", True, None),
    ("box", 366, 359, dict(kernel_size=1), "knn", True, None),
    ("box", 2, 65537, dict(kernel_size=15), "compat", False, (torch.float32, 4)),
    ("box", 65540, 2, dict(kernel_size=7), "knn", False, None),
    ("dense", 420, 313, dict(), "compat", False, None),
    ("dense", 520, 505, dict(kernel_size=7), "knn", True, (torch.float32, 5)),
    ("dense", 700, 375, dict(kernel_size=11, num_point_cloud_per_sp=9), "knn", False, None),
    ("hot", 384, 342, dict(), "compat", False, None),
    ("hot", 383, 343, dict(kernel_size=9), "knn", False, None),
    ("thin", 364, 364, dict(radius_threshold=0.02, kernel_size=9), "compat", False, None),
    ("thin", 364, 364, dict(t_intvl=0.0003, radius_threshold=0.02, kernel_size=9), "knn", False, None),
    ("thin", 364, 364, dict(t_intvl=-0.01), "knn", False, None),
    ("inside", 372, 353, dict(radius_threshold=0.05, kernel_size=6), "knn", False, None),
    ("far", 380, 346, dict(radius_threshold=0.01, kernel_size=8), "knn", False, None),
]


def build(kind, W, H, opts, dev, per_point, feat):
    pts, cam = scene(kind, W, H)
    opt = RenderOptions(**dict(dict(radius_threshold=0.012, num_point_cloud_per_sp=8), **opts))
    npts = NeuralPoints(pc_type="pc", points=to_dev(pts, dev))
    g = torch.Generator().manual_seed(5)
    rad = None
    if per_point:
        rad = (opt.radius_threshold * torch.exp(-2.3 * torch.rand(len(pts), generator=g))).to(dev)
    f = None
    if feat is not None:
        f = torch.randn((len(pts), feat[1]), generator=g).to(feat[0]).to(dev)
    return pts, cam, camera_spec(cam, dev), opt, npts, rad, f


def same(a, b, what):
    for k in a:
        assert np.array_equal(bits(a[k].cpu().numpy()), bits(b[k].cpu().numpy())), (what, k)


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}x{c[2]}-{c[4]}-k{c[3].get('kernel_size', 5)}")
def test_rows_equal_lane_sets(dev, case):
    kind, W, H, opts, mode, per_point, feat = case
    print("rows", case, flush=True)
    pts, cam, cs, opt, npts, rad, f = build(kind, W, H, opts, dev, per_point, feat)
    idx, depth, table = npts.pts2plane(cs, opt)
    for s_max in (None, 1, 5):
        kw = dict(radius=rad, mode=mode, feat=f, s_max=2 if rad is not None and s_max is None else s_max)
        same(npts.knn_sampling(cs, opt, idx, table, **kw), npts.knn_sampling(cs, opt, idx, table, cull=False, **kw),
             f"s_max {s_max}")
    dense = lambda cull, **kw: dict(zip("xitm", npts.render_image_hashtable_topk(  # noqa: E731
        cs, opt, idx, depth, table, mode=mode, cull=cull, **kw)))
    same(dense(True), dense(False), "dense")
    # lists: one wave per ray, with and without the point copy
    rays = torch.randint(-1, W * H + 1, (min(4 * W * H, 3000),), generator=torch.Generator().manual_seed(1))
    rays = rays.to(torch.int32).to(dev)
    kw = dict(radius=rad, mode=mode, feat=f, rays=rays, s_max=2)
    same(npts.knn_sampling(cs, opt, idx, table, **kw), npts.knn_sampling(cs, opt, idx, table, cull=False, **kw), "list")
    full = npts.knn_sampling(cs, opt, idx, table, radius=rad, mode=mode, feat=f, s_max=2)
    ok = (rays >= 0) & (rays < W * H)
    part = npts.knn_sampling(cs, opt, idx, table, **dict(kw, rays=rays[ok]))
    same(part, {k: v[rays[ok].long()] for k, v in full.items()}, "list against image")


@pytest.mark.parametrize("case", [CASES[1], CASES[7], CASES[12], CASES[18], CASES[28]], ids=lambda c: c[0])
def test_rows_oracle(dev, case):
    kind, W, H, opts, mode, _, _ = case
    pts, cam, cs, opt, npts, _, _ = build(kind, W, H, opts, dev, False, None)
    print("rows oracle", case, flush=True)
    idx, depth, table = npts.pts2plane(cs, opt)
    got = npts.render_image_hashtable_topk(cs, opt, idx, depth, table, mode=mode)
    oi, od, oh = oracle.pts2plane(pts, cam.w2c, cam.K, H, W)
    want = oracle.quick_sampling(pts, oracle.camera_from(cam), oracle.options_from(opt), oi, oh,
                                 mode=oracle.MODE_KNN if mode == "knn" else oracle.MODE_COMPAT)
    assert int(want[3].sum()) > 0
    for a, b in zip(got, want):
        assert np.array_equal(bits(a.cpu().numpy().reshape(b.shape)), bits(b))


@pytest.mark.parametrize("mode,W,H", [("compat", 100, 60), ("knn", 100, 60), ("compat", 368, 357)])
def test_rows_masked_table(dev, mode, W, H):
    """A table with pixels taken out: the buckets of a row are no longer one
    run of list positions."""
    _, _, cs, opt, npts, _, _ = build("box", W, H, {}, dev, False, None)
    idx, depth, table = npts.pts2plane(cs, opt)
    masked = table.clone()
    masked[(torch.rand(len(table), generator=torch.Generator().manual_seed(3)) < 0.3).to(dev)] = -1
    print("rows masked table", mode, W, H, flush=True)
    a = npts.knn_sampling(cs, opt, idx, masked, mode=mode)
    same(a, npts.knn_sampling(cs, opt, idx, masked, mode=mode, cull=False), "masked")
    assert int(a["n_samples"].sum()) > 0
