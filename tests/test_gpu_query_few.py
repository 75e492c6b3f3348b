"""The radius query's groups of four and eight lanes (few outputs, many rays)
against the oracle, entry for entry: the ray counts, windows and caps where the
group changes, with buckets that fill up and continue between steps."""
import numpy as np
import pytest

from epcq.epcq import RenderOptions
from test_gpu_query import query, scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,cap", [(1, 1), (1, 32), (1, 33), (2, 1), (2, 32), (3, 1), (3, 7), (3, 32), (3, 33), (4, 32)])
@pytest.mark.parametrize("R", [16383, 16384, 16399])
@pytest.mark.parametrize("kind", ["box", "hot"])
def test_small_windows(dev, kind, R, k, cap):
    W, H = 97, 65
    pts, cam = scene(kind, W, H)
    opt = RenderOptions(kernel_size=k, num_point_per_ray=cap, radius_threshold=0.02)
    rays = np.random.default_rng(R).integers(-3, W * H + 3, size=R).astype(np.int32)
    print("query few", kind, R, k, cap, flush=True)
    assert (query(dev, pts, cam, opt, None, rays) >= 0).any()


@pytest.mark.parametrize("k,cap", [(2, 3), (3, 5), (3, 32), (4, 1), (5, 32), (5, 33), (9, 2), (9, 32), (10, 5)])
@pytest.mark.parametrize("R", [131071, 131072, 131077])
@pytest.mark.parametrize("kind", ["box", "hot"])
def test_many_rays(dev, kind, R, k, cap):
    W, H = 97, 65
    pts, cam = scene(kind, W, H)
    opt = RenderOptions(kernel_size=k, num_point_per_ray=cap, radius_threshold=0.02)
    rays = np.random.default_rng(R).integers(-3, W * H + 3, size=R).astype(np.int32)
    print("query few, many rays", kind, R, k, cap, flush=True)
    assert (query(dev, pts, cam, opt, None, rays) >= 0).any()
