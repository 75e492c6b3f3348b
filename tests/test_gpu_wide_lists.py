"""Ray lists with windows of more than 256 lanes (kernel_size above 16): radii
that reach the window's last rows, against the oracle and the image's rows bit
for bit, whatever the list's length."""
import numpy as np
import pytest

from epcq import synth
from scenes import to_dev
from test_gpu_sampling import View, compact_vs_dense
from test_gpu_wave import dense_rays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,per_point", [(16, False), (17, False), (17, True), (20, False), (33, False)])
def test_wide_windows_of_listed_rays(dev, k, per_point):
    W, H = 90, 70
    pts = synth.box_scene(12_000, n_boxes=12, seed=3)
    cam = synth.look_at_camera([2.2, -2.4, 2.1], W, H, 1.39 * W)
    r = 0.45 * k * 3.9 / (1.39 * W)  # nearly half a window at the scene's distance
    rng = np.random.default_rng(k)
    radius = rng.uniform(0.5 * r, r, len(pts)).astype(np.float32) if per_point else None
    v = View(pts, cam, dev, radius=radius, kernel_size=k, radius_threshold=r, num_point_cloud_per_sp=8,
             num_sample_points_per_ray=2)
    rays = rng.integers(0, W * H, 700).astype(np.int32)
    uv = np.stack([rays % W, rays // W], axis=1).astype(np.int64)
    for mode in ("compat", "knn"):
        print(f"wide list k={k} {mode} per_point={per_point}", flush=True)
        part = compact_vs_dense(v, mode, rays=rays)
        compact_vs_dense(v, mode, rays=rays, cull=False)
        full = v.npts.knn_sampling(v.cs, v.opt, v.idx_d, v.hash_d, radius=v.radius_d, mode=mode)
        at = to_dev(rays, dev).long()
        for key in part:
            assert (part[key].cpu().numpy() == full[key][at].cpu().numpy()).all(), key
        if not per_point:
            dense_rays(v, mode, uv, min_live=100)
