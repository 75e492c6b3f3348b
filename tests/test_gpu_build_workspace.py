"""The build's two binned forms: 16-byte records, and arrays of their own in a
workspace too small for these; the same outputs, bit for bit, with runs that the
depth sort takes through the binned points as scratch."""
import numpy as np
import pytest
import torch

import epcq.csrc as C
from epcq import synth
from scenes import to_dev
from test_zz_no_alloc import run, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sort", [0, 1])
@pytest.mark.parametrize("n,W,H,hot", [(1, 1, 1, 0), (257, 9, 5, 0), (60_000, 97, 65, 0), (60_000, 97, 65, 5000),
                                       (300_000, 640, 480, 70_000)])
def test_smaller_workspace(dev, n, W, H, hot, sort):
    rng = np.random.default_rng(n)
    pts = synth.box_scene(max(n, 1000), n_boxes=12, seed=1)[:n]
    if hot:  # a pixel's run of `hot` points, in no depth order
        pts[:hot] = np.float32([0.01, 0.02, 0.03]) * rng.uniform(0.99, 1.01, (hot, 1)).astype(np.float32)
    cam = synth.look_at_camera([2.2, -2.4, 2.1], W, H, 1.39 * max(W, 48))
    xyz = to_dev(np.ascontiguousarray(pts, np.float32), dev)
    build = C._lib.epcq_build_hashtable
    full = C._lib.epcq_build_hashtable_workspace_size(n, H, W)
    small = full - 6 * n + 768  # 10 bytes per point instead of 16, and two more roundings to 256
    print("build workspace", n, W, H, hot, sort, full, small, flush=True)
    a = run(build, xyz, cam, sort, dev, torch.empty(full, dtype=torch.uint8, device=dev))
    b = run(build, xyz, cam, sort, dev, torch.empty(small, dtype=torch.uint8, device=dev))
    same(a, b)
