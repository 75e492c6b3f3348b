"""Performance cases of the epcq framework: what its users run, through its
public entry points, from the smallest call to the largest.

Kinds of case:
  build   NeuralPoints.pts2plane: projection, per-pixel point lists, hash table
  view    pts2plane + render_image_hashtable_topk: one image in the dense
          drop-in layout, as the reference's renderer samples it
  knn     pts2plane + knn_sampling: one image in the compact layout, with
          per-point radii, feature blending and wide windows
  rays    pts2plane + render_image_hashtable_topk(training_ray_index=...): the
          point search of one training step
  query   quick_query_for_nearby_point: the radius query of the point-search
          benchmark, on a table that is already built
  batch   MultiViewSampler: views of mixed resolution in one graph replay
  render  clamp_t + render and its backward: the compositing of a training
          step or of a whole image
  agg     Aggregator.forward: the MLPs over the neighbours of the live samples

Clouds, cameras and attributes are made on the GPU from the seed alone, with
the distributions of epcq.synth's scenes (points on boxes and a ground plane,
or on a sphere, with jitter; eyes on a sphere of radius 4).
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "hashpoint-code_amd"))

import epcq.csrc as C  # noqa: E402
from epcq import synth  # noqa: E402
from epcq.batch import MultiViewSampler  # noqa: E402
from epcq.epcq import Aggregator, CameraSpec, NeuralPoints, RenderOptions, clamp_t, render  # noqa: E402

DEV = "cuda:0"
RESOLUTIONS = synth.RESOLUTIONS


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest build: a 100k-point object, one small view; launches and
        # host time count
        {"name": "build-100k-400x400", "kind": "build", "scene": "sphere", "points": 100_000, "w": 400, "h": 400,
         "sort": False},
        # the largest build: a 20M-point scene at 1080p
        {"name": "build-20M-1080p", "kind": "build", "scene": "box200", "points": 20_000_000, "w": 1920, "h": 1080,
         "sort": False},
        # a renderer's image: 1M points, 800x800, 16 sample slots of 8
        # neighbours in the reference's dense layout
        {"name": "view-1M-800x800", "kind": "view", "scene": "box20", "points": 1_000_000, "w": 800, "h": 800,
         "radius": 0.005, "S": 16, "K": 8, "mode": "compat"},
        # nearest neighbours with blended fp32 features of an object at an odd
        # size
        {"name": "knn-307k-517x389-f16", "kind": "knn", "scene": "sphere", "points": 307_201, "w": 517, "h": 389,
         "k": 5, "radius": 0.01, "per_point": False, "K": 5, "feat": "f32", "F": 16},
        # the largest image: 20M points with radii of their own, the window
        # sized from the largest radius, 16 neighbours, 32 bf16 features
        {"name": "knn-20M-1080p-k15-bf16", "kind": "knn", "scene": "box200", "points": 20_000_000, "w": 1920,
         "h": 1080, "k": 15, "radius": 0.01, "per_point": True, "K": 16, "feat": "bf16", "F": 32},
        # a training step's point search: 4096 random rays of one view
        {"name": "rays-1M-800x800-4096", "kind": "rays", "scene": "box20", "points": 1_000_000, "w": 800, "h": 800,
         "radius": 0.005, "S": 16, "K": 8, "rays": 4096},
        # the radius query of the point-search benchmark: every ray of a small
        # image
        {"name": "query-200k-400x300", "kind": "query", "scene": "box20", "points": 200_000, "w": 400, "h": 300,
         "radius": 0.01, "cap": 256, "rays": 120_000},
        # serving and multi-view work: 24 views of mixed resolution of one
        # cloud, a captured graph replayed
        {"name": "batch-1M-24views", "kind": "batch", "points": 1_000_000, "views": 24, "first": 0,
         "radius": 0.005, "K": 8, "mode": "compat"},
        # compositing of one training step, forward and backward
        {"name": "render-4096x24", "kind": "render", "rays": 4096, "S": 24, "white_bg": False},
        # compositing of a whole image, forward and backward
        {"name": "render-640000x16", "kind": "render", "rays": 640_000, "S": 16, "white_bg": True},
        # the MLPs of one training batch: 4001 live samples of 5 neighbours
        {"name": "agg-4001x5", "kind": "agg", "samples": 4001, "K": 5},
        # the MLPs of a whole 800x800 image, two samples per ray
        {"name": "agg-1280000x8", "kind": "agg", "samples": 1_280_000, "K": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    w = _log(rng, lo, hi)
    return w, max(48, int(w * rng.choice([0.5625, 0.75, 1.0])) + rng.randrange(0, 4))


def _cloud(rng, w, h, lo, hi):
    """A point count for a w x h view: at most 40 points per pixel."""
    return min(_log(rng, lo, hi), 40 * w * h)


def draw(rng):
    kind = rng.choice(["build", "view", "knn", "rays", "query", "batch", "render", "agg"])
    scene = rng.choice(["sphere", "box20", "box80"])
    if kind == "build":
        w, h = _size(rng, 160, 1920)
        return {"kind": kind, "scene": scene, "points": _cloud(rng, w, h, 20_000, 18_000_000), "w": w, "h": h,
                "sort": rng.random() < 0.4}
    if kind == "view":
        w, h = _size(rng, 160, 800)
        return {"kind": kind, "scene": scene, "points": _cloud(rng, w, h, 50_000, 3_000_000), "w": w, "h": h,
                "radius": rng.uniform(0.004, 0.01), "S": rng.choice([8, 12, 16, 24]), "K": rng.choice([4, 8]),
                "mode": rng.choice(["compat", "knn"])}
    if kind == "knn":
        w, h = _size(rng, 160, 1920)
        k = rng.choice([3, 5, 7, 9, 11, 15])
        return {"kind": kind, "scene": scene, "points": _cloud(rng, w, h, 50_000, 12_000_000), "w": w, "h": h,
                "k": k, "radius": rng.uniform(0.004, 0.01), "per_point": rng.random() < 0.5,
                "K": rng.choice([1, 4, 5, 8, 12, 16, 32]), "feat": rng.choice(["none", "f32", "bf16"]),
                "F": rng.choice([8, 16, 19, 32])}
    if kind == "rays":
        w, h = _size(rng, 200, 1600)
        return {"kind": kind, "scene": scene, "points": _cloud(rng, w, h, 50_000, 5_000_000), "w": w, "h": h,
                "radius": rng.uniform(0.004, 0.01), "S": rng.choice([8, 16, 24]), "K": rng.choice([4, 8]),
                "rays": _log(rng, 256, 32768)}
    if kind == "query":
        w, h = _size(rng, 160, 800)
        return {"kind": kind, "scene": scene, "points": _cloud(rng, w, h, 20_000, 2_000_000), "w": w, "h": h,
                "radius": rng.uniform(0.004, 0.012), "cap": rng.choice([64, 100, 256]),
                "rays": min(_log(rng, 1024, 500_000), w * h)}
    if kind == "batch":
        return {"kind": kind, "points": _log(rng, 200_000, 1_000_000), "views": rng.randint(2, 20),
                "first": rng.randrange(5), "radius": rng.uniform(0.004, 0.007), "K": rng.choice([4, 8]), "mode": rng.choice(["compat", "knn"])}
    if kind == "render":
        S = rng.choice([2, 7, 8, 16, 24, 33, 64, 80])
        return {"kind": kind, "rays": min(_log(rng, 500, 1_200_000), 12_000_000 // S), "S": S,
                "white_bg": rng.random() < 0.5}
    K = rng.choice([1, 3, 4, 5, 8, 11, 16])
    return {"kind": kind, "samples": min(_log(rng, 700, 1_000_000), 8_000_000 // K), "K": K}


# ------------------------------------------------------------------ the inputs
def _gen(seed):
    return torch.Generator(DEV).manual_seed(seed)


def _normal(g, *shape):
    return torch.randn(shape, device=DEV, generator=g)


def _uniform(g, *shape):
    return torch.rand(shape, device=DEV, generator=g)


def _scene(name, n, seed):
    """[n, 3] float32 points on a sphere, or on random boxes and the ground
    plane by area (the distributions of synth.sphere_cloud / box_scene)."""
    g = _gen(seed)
    if name == "sphere":
        p = _normal(g, n, 3)
        return (p / p.norm(dim=1, keepdim=True) + 0.005 * _normal(g, n, 3)).contiguous()
    boxes = int(name[3:])
    sides = 0.1 + 0.4 * _uniform(g, boxes, 3)
    centres = 2.0 * _uniform(g, boxes, 3) - 1.0
    # faces: box b, normal axis a and sign s; the ground plane is the last
    box = torch.arange(boxes, device=DEV).repeat_interleave(6)
    axis = torch.arange(3, device=DEV).repeat_interleave(2).repeat(boxes)
    sign = torch.tensor([-1.0, 1.0], device=DEV).repeat(3 * boxes)
    other = sides[box].prod(dim=1) / sides[box, axis]
    cdf = torch.cumsum(torch.cat([other, torch.tensor([16.0], device=DEV)]).double(), 0)
    which = torch.searchsorted(cdf / cdf[-1], torch.rand(n, device=DEV, dtype=torch.float64, generator=g))
    which = which.clamp_max(6 * boxes)
    uv = _uniform(g, n, 3)
    f = which.clamp_max(6 * boxes - 1)
    p = centres[box[f]] + (uv - 0.5) * sides[box[f]]
    a = axis[f][:, None]
    face = centres[box[f]].gather(1, a) + 0.5 * sign[f][:, None] * sides[box[f]].gather(1, a)
    p.scatter_(1, a, face)
    plane = torch.stack([4.0 * uv[:, 0] - 2.0, 4.0 * uv[:, 1] - 2.0, torch.full_like(uv[:, 0], -1.0)], dim=1)
    p = torch.where((which == 6 * boxes)[:, None], plane, p)
    return (p + 0.002 * _normal(g, n, 3)).contiguous()


def _camera(rnd, w, h):
    d = [rnd.gauss(0.0, 1.0) for _ in range(3)]
    n = math.sqrt(sum(x * x for x in d)) or 1.0
    return synth.look_at_camera([4.0 * x / n for x in d], w, h, synth.nerf_focal(w))


def _spec(cam):
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    return CameraSpec(c2w=t(cam.c2w), w2c=t(cam.w2c), K=t(cam.K), fx=cam.fx, fy=cam.fy, cx=cam.cx, cy=cam.cy,
                      width=cam.width, height=cam.height)


def _resolutions(case):
    """The views' sizes: the resolution classes in turn."""
    return [RESOLUTIONS[(case["first"] + i) % len(RESOLUTIONS)] for i in range(case["views"])]


def _options(case):
    return RenderOptions(kernel_size=case.get("k", 5), radius_threshold=case["radius"],
                         num_sample_points_per_ray=case.get("S", 16), num_point_cloud_per_sp=case.get("K", 8),
                         num_point_per_ray=case.get("cap", 256))


def _aggregator_inputs(M, K, seed):
    """What FeatureQuery hands over for M live samples: neighbours within about
    0.01 of their sample, nine in ten valid, zeros in the place of the others."""
    g = _gen(seed)
    sp = 2.0 * _uniform(g, M, 3) - 1.0
    valid = _uniform(g, M, K) < 0.9
    valid[:, 0] = True
    z = ~valid[..., None]
    pc = (sp[:, None, :] + 0.01 * _normal(g, M, K, 3)).masked_fill_(z, 0.0)
    rgb = _uniform(g, M, K, 3).masked_fill_(z, 0.0)
    d = _normal(g, M, K, 3)
    d = (d / d.norm(dim=-1, keepdim=True)).masked_fill_(z, 0.0)
    feat = _normal(g, M, K, 32).masked_fill_(z, 0.0)
    rays = _normal(g, M, 3)
    return pc, rgb, d, feat, sp, valid, rays / rays.norm(dim=-1, keepdim=True)


def prepare(case, seed):
    kind = case["kind"]
    rnd = random.Random(seed)
    s = {"kind": kind}
    if kind == "agg":
        torch.manual_seed(seed)  # weights of the module's own initialisation
        mod = Aggregator().to(DEV)
        g = _gen(seed + 1)
        with torch.no_grad():
            for p in mod.parameters():
                if p.dim() == 1:
                    p.copy_(0.1 * _normal(g, *p.shape))
            mod.packed_params()
        s["mod"] = mod
        s["inputs"] = _aggregator_inputs(case["samples"], case["K"], seed)
        s["mask"] = torch.ones((case["samples"], 1), dtype=torch.bool, device=DEV)
        return s
    if kind == "render":
        g = _gen(seed)
        R, S = case["rays"], case["S"]
        s["t"] = 2.0 + 4.0 * _uniform(g, R, 1) + torch.cumsum(0.012 * _uniform(g, R, S), dim=1)
        s["sigma"] = (-20.0 * torch.log1p(-_uniform(g, R, S))).requires_grad_()
        s["rgb"] = _uniform(g, R, S, 3).requires_grad_()
        s["grad"] = _normal(g, R, 3)
        s["white_bg"] = case["white_bg"]
        return s
    if kind == "batch":
        xyz = _scene("box20", case["points"], seed)
        # the launch shape that the autotuner finds for such batches
        tuning = {"tile_w": 16, "tile_h": 16, "tile_cap": 1536, "flags": C.TUNE_XCD_ORDER, "heavy": 256}
        sampler = MultiViewSampler(_options(case), mode=case["mode"], max_views=case["views"], tuning=tuning,
                                   device=DEV)
        sampler.set_views([(xyz, _camera(rnd, w, h)) for w, h in _resolutions(case)])
        sampler.capture()
        s["sampler"] = sampler
        return s
    w, h = case["w"], case["h"]
    xyz = _scene(case["scene"], case["points"], seed)
    s["points"] = NeuralPoints(pc_type="pc", points=xyz)
    s["cam"] = _spec(_camera(rnd, w, h))
    if kind == "build":
        s["opt"] = RenderOptions()
        s["sort"] = case["sort"]
        return s
    s["opt"] = _options(case)
    g = _gen(seed + 1)
    if kind == "view":
        s["mode"] = case["mode"]
    elif kind == "knn":
        s["radius"] = s["feat"] = None
        s["r_max"] = case["radius"]
        if case["per_point"]:  # log-uniform over a factor of ten
            s["radius"] = case["radius"] * torch.exp(math.log(0.1) * _uniform(g, case["points"]))
        if case["feat"] != "none":
            dtype = torch.bfloat16 if case["feat"] == "bf16" else torch.float32
            s["feat"] = _normal(g, case["points"], case["F"]).to(dtype)
    elif kind == "rays":
        s["uv"] = torch.stack([torch.randint(0, w, (case["rays"],), device=DEV, generator=g),
                               torch.randint(0, h, (case["rays"],), device=DEV, generator=g)], dim=1)
    elif kind == "query":
        s["rays"] = torch.randperm(w * h, device=DEV, generator=g)[:case["rays"]].to(torch.int32)
        s["table"] = s["points"].pts2plane(s["cam"], s["opt"])
    return s


# -------------------------------------------------------------------- the work
def run(s):
    kind = s["kind"]
    if kind == "build":
        return s["points"].pts2plane(s["cam"], s["opt"], sort=s["sort"])
    if kind == "agg":
        with torch.no_grad():
            pc, rgb, d, feat, sp, valid, rays = s["inputs"]
            return s["mod"](pc, rgb, d, feat, sp, valid, s["mask"], rays)
    if kind == "render":
        deltas = clamp_t(s["t"])
        colours = render(deltas, s["sigma"], s["rgb"], white_bg=s["white_bg"])
        return (colours.detach(),) + torch.autograd.grad(colours, (s["sigma"], s["rgb"]), s["grad"])
    if kind == "batch":
        sampler = s["sampler"]
        sampler.replay()
        out, _ = sampler.batch_outputs()
        tables = []
        for i in range(len(sampler.views)):
            o = sampler.view_outputs(i)
            tables.append((o["sorted_idx"], o["hash"]))
        return out, tables
    points, cam, opt = s["points"], s["cam"], s["opt"]
    if kind == "query":
        idx, _, table = s["table"]
        return C.quick_query_for_nearby_point(points._to_cpp(), cam._to_cpp(), opt._to_cpp(), idx, table, s["rays"])
    idx, depth, table = points.pts2plane(cam, opt)
    if kind == "view":
        return points.render_image_hashtable_topk(cam, opt, idx, depth, table, mode=s["mode"])
    if kind == "rays":
        return points.render_image_hashtable_topk(cam, opt, idx, depth, table, training_ray_index=s["uv"])
    return points.knn_sampling(cam, opt, idx, table, radius=s["radius"], feat=s["feat"], r_max=s["r_max"])


def work(case):
    """Bytes: every input read once and every output written once (every
    neighbour's point and features are counted once per point of the cloud);
    flops: of the MLPs, on the neighbours that are valid."""
    kind = case["kind"]
    if kind == "agg":
        M, K = case["samples"], case["K"]
        pairs = M * (1 + 0.9 * (K - 1))
        flops = pairs * 2 * (284 * 256 + 256 * 256 + 263 * 256 + 256 * 256 + 256)
        flops += M * 2 * (280 * 128 + 2 * 128 * 128 + 128 * 3)
        return {"bytes": M * K * (41 * 4 + 1) + M * (24 + 1 + 16), "flops": flops}
    if kind == "render":
        R, S = case["rays"], case["S"]
        # t, sigma, rgb and the colours' gradient in; colours and gradients out
        return {"bytes": R * (20 * S + 12 + 12 + 16 * S), "flops": R * S * 60}
    n = case["points"]
    if kind == "batch":
        pixels = sum(w * h for w, h in _resolutions(case))
        per_ray = 4 + 2 * (4 + (4 if case["mode"] == "compat" else 12) * case["K"])
        return {"bytes": case["views"] * 16 * n + pixels * (8 + per_ray), "flops": 0}
    pixels = case["w"] * case["h"]
    build = 20 * n + 8 * pixels
    if kind == "build":
        return {"bytes": build, "flops": 60 * n}
    if kind == "query":
        return {"bytes": 16 * n + 8 * pixels + case["rays"] * 4 * (1 + case["cap"]), "flops": 0}
    if kind == "view":
        return {"bytes": build + pixels * case["S"] * (17 + 4 * case["K"]), "flops": 0}
    if kind == "rays":
        return {"bytes": build + case["rays"] * (16 + case["S"] * (17 + 4 * case["K"])), "flops": 0}
    F = 0 if case["feat"] == "none" else case["F"]
    out = 4 + 2 * (4 + case["K"] * (16 if F else 12) + 4 * F)
    feat = F * (2 if case["feat"] == "bf16" else 4)
    return {"bytes": build + n * ((4 if case["per_point"] else 0) + feat) + pixels * out, "flops": 0}


# ----------------------------------------------------------- 64-bit references
def _exact_render(s):
    """clamp_t and alpha compositing in float64.  Which intervals are clamped
    is decided on the float32 differences: a threshold has no nearby value."""
    t = s["t"]
    d = t[:, 1:] - t[:, :-1]
    vsize = torch.tensor(0.004, device=t.device).item()
    clamped = (d < 1e-8) | (d > 2 * vsize)
    d = torch.where(clamped, torch.full_like(d, 0.0).double() + 0.004, t[:, 1:].double() - t[:, :-1].double())
    deltas = torch.cat([d, torch.full_like(d[:, :1], 0.004)], dim=1)
    sigma = s["sigma"].detach().double().requires_grad_()
    rgb = s["rgb"].detach().double().requires_grad_()
    opacity = 1.0 - torch.exp(-sigma * deltas)
    trans = torch.cumprod(1.0 - opacity + 1e-10, dim=1)
    trans = torch.cat([torch.ones_like(trans[:, :1]), trans[:, :-1]], dim=1)
    out = (rgb * (opacity * trans)[..., None]).sum(dim=1)
    if s["white_bg"]:
        out = out + trans[:, -1:]
    return (out.detach(),) + torch.autograd.grad(out, (sigma, rgb), s["grad"].double())


def _encode(x, freqs):
    p = (x[..., None] * (2.0 ** torch.arange(freqs, dtype=x.dtype, device=x.device))).flatten(-2)
    return torch.stack([torch.sin(p), torch.cos(p)], dim=-1).flatten(-2)


def _exact_agg(s):
    par = {k: v.detach().double() for k, v in s["mod"].state_dict().items()}
    act = torch.nn.functional.leaky_relu

    def linear(x, name):
        return x @ par[name + ".weight"].t() + par[name + ".bias"]

    alphas, colours = [], []
    M = s["inputs"][0].shape[0]
    for i in range(0, M, 40_000):
        pc, rgb, d, feat, sp, valid, rays = [x[i:i + 40_000] for x in s["inputs"]]
        pc, rgb, d, feat, sp, rays = [x.double() for x in (pc, rgb, d, feat, sp, rays)]
        dist = pc - sp[:, None, :]
        power = pc.square() - sp[:, None, :].square()
        w = valid.double() / (dist.norm(dim=-1) + 1e-6)
        w = w / (w.sum(dim=-1, keepdim=True) + 1e-6)
        h = torch.cat([feat, _encode(feat, 3), _encode(torch.cat([dist, power], dim=-1), 5)], dim=-1)
        h = act(linear(act(linear(h, "block1.0")), "block1.2"))
        rd = rays[:, None, :]
        h = torch.cat([h, rgb, d - rd, (d * rd).sum(dim=-1, keepdim=True)], dim=-1)
        h = act(linear(act(linear(h, "block3.0")), "block3.2"))
        a = torch.nn.functional.softplus(linear(h, "alpha_branch.0") - 1.0)
        alphas.append((a[..., 0] * w).sum(dim=-1))
        x = torch.cat([(h * w[..., None]).sum(dim=-2), _encode(rays, 4)], dim=-1)
        for name in ("color_branch.0", "color_branch.2", "color_branch.4"):
            x = act(linear(x, name))
        colours.append(torch.sigmoid(linear(x, "color_branch.6")) * 1.002 - 0.001)
    return torch.cat(alphas)[:, None], torch.cat(colours)[:, None, :]


def exact(case, seed):
    """64-bit results of the compositing and of the MLPs.  The searches return
    point indices, and depths picked by comparisons that are defined on 32-bit
    values: they have no 64-bit counterpart."""
    if case["kind"] == "render":
        return _exact_render(prepare(case, seed))
    if case["kind"] == "agg":
        return _exact_agg(prepare(case, seed))
    return None
