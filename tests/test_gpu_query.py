"""The radius query's groups of lanes against the oracle, entry for entry: the
window sizes and ray counts where the group changes, buckets that fill up, end
and continue between steps, caps inside a step, and pixels outside the image."""
import numpy as np
import pytest
import torch

import epcq.csrc as C
from epcq import synth
from epcq.epcq import NeuralPoints, RenderOptions
from oracle import oracle
from scenes import camera_spec, to_dev

pytestmark = pytest.mark.gpu


def scene(kind, W, H):
    rng = np.random.default_rng(7)
    cam = synth.look_at_camera([2.2, -2.4, 2.1], W, H, 1.39 * W)
    pts = synth.box_scene(60_000, n_boxes=12, seed=1)
    if kind == "hot":  # a few pixels with thousands of points each, most of them hits
        at = rng.uniform(-0.5, 0.5, (6, 3))
        hot = (np.repeat(at, 3000, axis=0) + rng.normal(0, 1e-3, (18_000, 3))).astype(np.float32)
        pts = np.concatenate([pts[:20_000], hot])
    return np.ascontiguousarray(pts, np.float32), cam


def query(dev, pts, cam, opt, table, rays):
    cs, npts = camera_spec(cam, dev), NeuralPoints(pc_type="pc", points=to_dev(pts, dev))
    if table is None:
        idx, _, h = npts.pts2plane(cs, opt)
    else:
        idx, h = (to_dev(t, dev) for t in table)
    got = C.quick_query_for_nearby_point(npts._to_cpp(), cs._to_cpp(), opt._to_cpp(), idx, h, to_dev(rays, dev))
    oi, oh = idx.cpu().numpy(), h.cpu().numpy().reshape(-1, 2)
    want = oracle.quick_query(pts, oracle.camera_from(cam), oracle.options_from(opt), oi, oh, rays)
    got = got.cpu().numpy()
    np.testing.assert_array_equal(got, want.reshape(got.shape))
    return got


@pytest.mark.parametrize("R", [1, 7, 16383, 16384, 16387])
@pytest.mark.parametrize("k,cap", [(1, 3), (5, 100), (5, 33), (6, 256), (9, 64), (29, 128)])
@pytest.mark.parametrize("kind", ["box", "hot"])
def test_query_groups(dev, kind, k, cap, R):
    W, H = 97, 65
    pts, cam = scene(kind, W, H)
    opt = RenderOptions(kernel_size=k, num_point_per_ray=cap, radius_threshold=0.02)
    rays = np.random.default_rng(R).integers(-3, W * H + 3, size=R).astype(np.int32)
    if R <= 7:
        rays[:] = np.abs(rays) % W + (H // 2) * W
    print("query", kind, k, cap, R, flush=True)
    got = query(dev, pts, cam, opt, None, rays)
    assert R <= 7 or (got >= 0).any()


def test_query_bucket_of_many_points(dev):
    """A bucket of more than 2^24 points between small ones."""
    W = H = 9
    n, big = (1 << 24) + 5000, (1 << 24) + 1000
    cam = synth.look_at_camera([0.0, -4.0, 0.0], W, H, 12.0)
    pts = np.full((n, 3), 50.0, np.float32)
    hits = np.concatenate([np.arange(0, 40), 1000 + np.array([3, 70, 1 << 20, 1 << 24, big - 1]),
                           1000 + big + np.arange(5, 25)])
    pts[hits] = np.random.default_rng(2).uniform(-0.01, 0.01, (len(hits), 3))
    table = np.full((W * H, 2), -1, np.int32)
    table[4 * W + 3] = (0, 1000)
    table[4 * W + 4] = (1000, big)
    table[4 * W + 5] = (1000 + big, n - 1000 - big)
    opt = RenderOptions(kernel_size=3, num_point_per_ray=64, radius_threshold=1.0)
    rays = np.array([4 * W + 4, 3 * W + 4, 0, 4 * W + 6], np.int32)
    print("query bucket of", big, flush=True)
    got = query(dev, pts, cam, opt, (np.arange(n, dtype=np.int32), table), rays)
    assert (got[0] >= 0).sum() == 32 + 5 + 20
