"""Workspaces of the sizes that the library took before its 16-byte records and
candidate bounds: the public calls take them and give the same outputs, bit for
bit; what is smaller still is refused by the build."""
import numpy as np
import pytest
import torch

import epcq.csrc as C
from epcq import synth
from epcq.epcq import NeuralPoints, RenderOptions
from scenes import bits, camera_spec, to_dev

pytestmark = pytest.mark.gpu


def up(n):
    return (n + 255) // 256 * 256


def smallest_build(n, H, W):
    """Index, depth and pixel in arrays of their own, in place of the records."""
    return C.build_hashtable_workspace_size(n, H, W) - up(16 * n) + 2 * up(4 * n) + up(2 * n)


def scene(n, W, H, dev):
    cam = synth.look_at_camera([2.2, -2.4, 2.1], W, H, 1.39 * max(W, 48))
    pts = synth.box_scene(max(n, 1000), n_boxes=12, seed=1)[:n]
    return NeuralPoints(pc_type="pc", points=to_dev(np.ascontiguousarray(pts, np.float32), dev)), camera_spec(cam, dev)


def same(a, b):
    for x, y in zip(a, b):
        assert np.array_equal(bits(x.cpu().numpy()), bits(y.cpu().numpy()))


@pytest.mark.parametrize("sort", [False, True])
@pytest.mark.parametrize("n,W,H", [(257, 9, 5), (60_000, 97, 65), (300_001, 640, 480)])
def test_build_takes_ten_bytes_per_point(dev, n, W, H, sort):
    npts, cs = scene(n, W, H, dev)
    opt = RenderOptions()
    small = smallest_build(n, H, W)
    assert small < C.build_hashtable_workspace_size(n, H, W)
    print("build workspace", n, W, H, sort, small, flush=True)
    want = npts.pts2plane(cs, opt, sort=sort)
    same(npts.pts2plane(cs, opt, sort=sort, workspace=torch.empty(small, dtype=torch.uint8, device=dev)), want)
    with pytest.raises(RuntimeError, match="build_hashtable: workspace too small"):
        npts.pts2plane(cs, opt, sort=sort, workspace=torch.empty(small - 1, dtype=torch.uint8, device=dev))


@pytest.mark.parametrize("offset", [4, 8, 12])
def test_build_takes_a_workspace_at_any_word(dev, offset):
    n, W, H = 60_000, 97, 65
    npts, cs = scene(n, W, H, dev)
    opt = RenderOptions()
    print("build workspace at", offset, flush=True)
    for sort in (False, True):
        for size in (smallest_build(n, H, W), C.build_hashtable_workspace_size(n, H, W)):
            ws = torch.empty(offset + size, dtype=torch.uint8, device=dev)[offset:]
            same(npts.pts2plane(cs, opt, sort=sort, workspace=ws), npts.pts2plane(cs, opt, sort=sort))


@pytest.mark.parametrize("W,H,n", [(97, 65, 60_000), (390, 350, 150_001)])
def test_samplers_take_any_workspace(dev, monkeypatch, W, H, n):
    """Images and ray lists, with each part of the workspace just there and just
    missing: candidate bounds, radii, point copy, cones."""
    npts, cs = scene(n, W, H, dev)
    opt = RenderOptions(radius_threshold=0.012, num_point_cloud_per_sp=8, kernel_size=5)
    idx, depth, table = npts.pts2plane(cs, opt)
    g = torch.Generator().manual_seed(2)
    rays = torch.randint(0, W * H, (4000,), generator=g).to(torch.int32).to(dev)
    radius = (0.012 * torch.exp(-2.3 * torch.rand(n, generator=g))).to(dev)

    def calls():
        out = list(npts.render_image_hashtable_topk(cs, opt, idx, depth, table))
        for kw in (dict(), dict(radius=radius, s_max=2), dict(rays=rays), dict(rays=rays, radius=radius, s_max=2)):
            out += npts.knn_sampling(cs, opt, idx, table, mode="knn", **kw).values()
        return out

    cones = up(16 * H * W) + up(8 * H * W)
    points, radii = cones + up(16 * n), cones + up(16 * n) + 4 * n
    full = C._lib.epcq_sampling_workspace_size(n, H, W)
    sizes = [full, full - 1, radii, radii - 1, points, points - 1, cones, cones - 1]
    assert sizes == sorted(sizes, reverse=True)
    monkeypatch.setattr(C, "_workspace", lambda *a: None)
    want = calls()
    assert int(want[3].sum()) > 1000
    for size in sizes:
        print("sampler workspace", W, H, n, size, flush=True)
        monkeypatch.setattr(C, "_workspace", lambda *a: torch.empty(size, dtype=torch.uint8, device=dev))
        same(calls(), want)
