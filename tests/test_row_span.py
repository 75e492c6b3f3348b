"""Tables whose rows are not one run of the point list (buckets moved, shared or
taken out): what the tiled samplers stage of them, on the host under the
sanitizers, and every form of the samplers on them against the oracle."""
import os
import shutil
import subprocess

import numpy as np
import pytest
import torch

import epcq.csrc as C
from epcq import synth
from epcq.epcq import NeuralPoints, RenderOptions
from oracle import oracle
from scenes import bits, camera_spec, to_dev

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "sanitize")


def test_row_spans_on_the_host():
    if not os.path.exists("/opt/rocm/bin/hipcc") or not shutil.which("make"):
        pytest.skip("needs hipcc")
    subprocess.run(["make", "-s", "-C", HERE, "_build/row_span_driver"], check=True, capture_output=True, text=True)
    res = subprocess.run([os.path.join(HERE, "_build", "row_span_driver")], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0 and "ok" in res.stdout, res.stdout + res.stderr


def tables(idx, table, rng):
    """(name, sorted_idx, hash) of the same buckets, laid out otherwise."""
    full = np.flatnonzero(table[:, 1] > 0)

    def laid(order):
        out, t, at = np.full_like(idx, -1), table.copy(), 0
        for p in order:
            s, n = table[p]
            out[at:at + n] = idx[s:s + n]
            t[p] = at, n
            at += n
        return out, t

    yield ("reversed",) + laid(full[::-1])
    yield ("moved",) + laid(rng.permutation(full))
    shared = table.copy()
    shared[rng.choice(full, len(full) // 3)] = table[rng.choice(full, len(full) // 3)]
    yield "shared", idx, shared
    holes, gone = idx.copy(), table.copy()  # pixels taken out, with their indices
    for p in rng.choice(full, len(full) // 3, replace=False):
        s, n = table[p]
        holes[s:s + n] = -1
        gone[p] = -1
    yield "holes", holes, gone


@pytest.mark.gpu
@pytest.mark.parametrize("W,H,k,live,per_point", [(70, 50, 5, 2, False), (96, 64, 9, 2, True), (60, 45, 17, 2, False),
                                                  (130, 70, 4, 16, False), (368, 357, 5, 2, False)])
def test_tables_in_any_order(dev, W, H, k, live, per_point):
    rng = np.random.default_rng(W)
    pts = synth.box_scene(20_000, n_boxes=12, seed=3)
    cam = synth.look_at_camera([2.2, -2.4, 2.1], W, H, 1.39 * W)
    opt = RenderOptions(kernel_size=k, radius_threshold=0.02, num_point_cloud_per_sp=8,
                        **(dict(sdf2weight_gaussian_gamma=0.2, sdf2weight_gaussian_alpha=0.01) if live > 2 else {}))
    assert C.max_live_samples(opt, opt.radius_threshold) == live
    rad = (0.02 * np.exp(-1.5 * rng.random(len(pts)))).astype(np.float32) if per_point else None
    cs, npts = camera_spec(cam, dev), NeuralPoints(pc_type="pc", points=to_dev(pts, dev))
    oi, _, oh = oracle.pts2plane(pts, cam.w2c, cam.K, H, W)
    rays = rng.permutation(W * H)[:500].astype(np.int32)
    for name, idx, table in tables(oi, oh, rng):
        want = oracle.quick_sampling(pts, oracle.camera_from(cam), oracle.options_from(opt), idx, table,
                                     mode=oracle.MODE_KNN, radius=rad)
        xyz, nb, t, mask = want
        assert int(mask.sum()) > 300
        i_d, h_d = to_dev(idx, dev), to_dev(table, dev)
        for form, kw in [("bounds", {}), ("none", dict(cull=False)), ("list", dict(rays=to_dev(rays, dev))),
                         ("list, none", dict(rays=to_dev(rays, dev), cull=False))]:
            print("table", name, W, H, k, form, flush=True)
            o = npts.knn_sampling(cs, opt, i_d, h_d, mode="knn", s_max=live,
                                  radius=None if rad is None else to_dev(rad, dev), **kw)
            at = rays if "rays" in kw else slice(None)
            assert np.array_equal(o["n_samples"].cpu().numpy(), mask[at].sum(1)), (name, form)
            assert np.array_equal(o["nb_idx"].cpu().numpy(), nb[at][:, :live]), (name, form)
            assert np.array_equal(bits(o["sample_t"].cpu().numpy()), bits(t[at][:, :live])), (name, form)
        if rad is None:
            for cull in (True, False):
                print("table", name, W, H, k, "dense", cull, flush=True)
                got = npts.render_image_hashtable_topk(cs, opt, i_d, None, h_d, mode="knn", cull=cull)
                for a, b in zip(got, want):
                    assert np.array_equal(bits(a.cpu().numpy().reshape(b.shape)), bits(b)), (name, cull)
