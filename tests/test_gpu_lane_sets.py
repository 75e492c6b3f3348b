"""The lane-set kernels with their cones, staging and deferral on full images,
for the options and sizes that the row-run sampler takes by itself: calls with
a workspace of the size from before the candidate bounds, against the oracle
bit for bit."""
import pytest
import torch

import epcq.csrc as C
from epcq import autotune, synth
from test_gpu_sampling import View, check_dense, compact_vs_dense
from test_gpu_tunings import dense_view, name, tunings  # noqa: F401  (a fixture)
from test_gpu_wave import heavy_threshold
from test_gpu_wide_window import launch_shape

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def former_workspace(monkeypatch):
    """The samplers' workspace without the candidate bounds: cones, points and
    radii."""
    def up(n):
        return (n + 255) // 256 * 256

    def workspace(n, H, W, device, cull):
        if not cull:
            return None
        size = up(16 * H * W) + up(8 * H * W) + up(16 * n) + 4 * n
        assert size < C._lib.epcq_sampling_workspace_size(n, H, W)
        return torch.empty(size, dtype=torch.uint8, device=device)

    monkeypatch.setattr(C, "_workspace", workspace)


@pytest.mark.parametrize("tuning", tunings(), ids=name)
def test_tunings(dev, dense_view, tuning):  # noqa: F811
    old = C.get_tuning()
    print(f"lane sets, tuning {name(tuning)}", flush=True)
    try:
        autotune.apply(tuning)
        check_dense(dense_view, "compat")
        check_dense(dense_view, "knn")
    finally:
        C.set_tuning(**old)


@pytest.mark.parametrize("k", [9, 11, 15, 16])
@pytest.mark.parametrize("heavy", [0, 1])
def test_wide_window(dev, k, heavy):
    pts = synth.box_scene(300_000, n_boxes=20, seed=8)
    cam = synth.look_at_camera([2.0, -2.6, 1.9], 120, 90, synth.nerf_focal(120) * 2.0)
    v = View(pts, cam, dev, kernel_size=k, radius_threshold=0.012, num_point_cloud_per_sp=8)
    for mode in ("compat", "knn"):
        print(f"lane sets, wide window k={k} {mode} heavy={heavy}", flush=True)
        with heavy_threshold(heavy):
            check_dense(v, mode)
            compact_vs_dense(v, mode)


@pytest.mark.parametrize("cap,heavy", [(6000, 0), (1024, 0), (1024, 1)])
def test_staging_capacity_per_point_radius(dev, cap, heavy):
    pts = synth.box_scene(250_000, n_boxes=20, seed=11)
    radius = synth.log_uniform_radius(len(pts), seed=12, lo=2e-3, hi=2e-2)
    cam = synth.look_at_camera([2.4, 2.0, 1.8], 96, 80, synth.nerf_focal(96) * 2.0)
    v = View(pts, cam, dev, radius=radius, kernel_size=15, radius_threshold=0.02, num_point_cloud_per_sp=16)
    print(f"lane sets, k=15 staging cap={cap} heavy={heavy}", flush=True)
    with launch_shape(tile_w=16, tile_h=16, tile_cap=cap, heavy=heavy):
        check_dense(v, "knn")
        compact_vs_dense(v, "knn")


@pytest.mark.parametrize("kw", [
    dict(kernel_size=3, radius_threshold=0.02, num_point_cloud_per_sp=4),
    dict(kernel_size=7, radius_threshold=0.05, num_point_cloud_per_sp=12, num_sample_points_per_ray=4),
    dict(kernel_size=5, radius_threshold=0.04, t_intvl=0.001, num_point_cloud_per_sp=8),
    dict(kernel_size=1, radius_threshold=0.05, num_point_cloud_per_sp=3),
])
@pytest.mark.parametrize("heavy", [0, 1, 64])
def test_wave_form(dev, kw, heavy):
    pts = synth.sphere_cloud(40_000, seed=5)
    cam = synth.look_at_camera([0.3, -3.5, 0.4], 90, 70, 110.0)
    v = View(pts, cam, dev, **kw)
    feat = torch.randn(len(pts), 16, generator=torch.Generator().manual_seed(1)).to(dev)
    for mode in ("compat", "knn"):
        print(f"lane sets, wave form {mode} heavy={heavy} {kw}", flush=True)
        with heavy_threshold(heavy):
            check_dense(v, mode)
            compact_vs_dense(v, mode, feat=feat)


def test_wave_form_per_point_radius_k16(dev):
    pts = synth.box_scene(300_000, n_boxes=40, seed=8)
    radius = synth.log_uniform_radius(len(pts), seed=9)
    cam = synth.look_at_camera([2.0, -2.0, 3.0], 320, 180, 444.0)
    v = View(pts, cam, dev, radius=radius, kernel_size=7, radius_threshold=0.01, num_point_cloud_per_sp=16)
    feat = torch.randn(len(pts), 32, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).to(dev)
    print("lane sets, per-point radius K=16 + bf16 features", flush=True)
    with heavy_threshold(1):
        compact_vs_dense(v, "knn", feat=feat)


def test_former_workspace_equals_the_present_one(dev, monkeypatch):
    """One image per form of the row runs: the smaller workspace gives the same
    outputs bit for bit."""
    for W, H, n in ((200, 150, 200_000), (640, 400, 300_000)):
        pts = synth.box_scene(n, n_boxes=12, seed=2)
        cam = synth.look_at_camera([2.2, -2.4, 2.1], W, H, 1.39 * W)
        v = View(pts, cam, dev, radius_threshold=0.012, num_point_cloud_per_sp=8)
        small = v.npts.knn_sampling(v.cs, v.opt, v.idx_d, v.hash_d)
        assert C.sampling_form(v.opt, n, H, W) != C.FORM_LANE_SETS
        with monkeypatch.context() as m:
            m.setattr(C, "_workspace", lambda n, H, W, device, cull: torch.empty(
                C._lib.epcq_sampling_workspace_size(n, H, W), dtype=torch.uint8, device=device))
            full = v.npts.knn_sampling(v.cs, v.opt, v.idx_d, v.hash_d)
        for key in full:
            assert torch.equal(small[key].view(torch.int32), full[key].view(torch.int32)), key
