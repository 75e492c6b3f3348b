"""Which form a sampler call takes, and that the autotuner varies only what the
form reads (host only)."""
import epcq.csrc as C
from epcq import autotune
from epcq.epcq import RenderOptions


def form(n, W, H, rays=-1, live=None, compact=True, ws=None, **opt):
    return C.sampling_form(RenderOptions(**opt), n, H, W, live=live, compact=compact, rays=rays, workspace_bytes=ws)


def test_forms():
    assert form(1_000_000, 800, 800) == C.FORM_ROW_TILES
    assert form(1_000_000, 800, 800, compact=False) == C.FORM_ROW_TILES
    assert form(1_000_000, 200, 150) == C.FORM_ROW_WAVES
    # not over rows: no workspace, one of the former size, wide windows, more live samples
    full = C._lib.epcq_sampling_workspace_size(1_000_000, 800, 800)
    for kw in (dict(ws=0), dict(ws=full - 1), dict(kernel_size=17), dict(live=3),
               dict(sdf2weight_gaussian_gamma=0.2, sdf2weight_gaussian_alpha=0.01)):
        assert form(1_000_000, 800, 800, **kw) == C.FORM_LANE_SETS, kw
    # lists by their length
    old = C.get_tuning()
    try:
        C.set_tuning(**dict(old, list_wave=100))
        assert form(1_000_000, 800, 800, rays=100, ws=0) == C.FORM_ROW_WAVES
        assert form(1_000_000, 800, 800, rays=101) == C.FORM_LANE_SETS
    finally:
        C.set_tuning(**old)


def test_autotuner_varies_what_the_form_reads(monkeypatch):
    monkeypatch.setattr(autotune.torch.cuda, "get_device_name", lambda: "none")
    monkeypatch.setattr(autotune, "time_ms", lambda fn, **kw: fn())
    monkeypatch.setattr(autotune, "_cache", {"": 0})
    seen = []

    def run(t):  # every other setting is faster than the default
        seen.append(t)
        return 2.0 if t == autotune.DEFAULT else 1.0 + 0.01 * len(seen)

    best, _ = autotune.tune("waves", run, **autotune.knobs(C.FORM_ROW_WAVES))
    assert best == autotune.DEFAULT and not seen
    best, _ = autotune.tune("tiles", run, **autotune.knobs(C.FORM_ROW_TILES, heavy=(128, 512, 0)))
    assert {k: v for k, v in best.items() if k != "heavy"} == {k: v for k, v in autotune.DEFAULT.items() if k != "heavy"}
    assert sorted({t["heavy"] for t in seen}) == [0, 128, 512]
    best, _ = autotune.tune("lanes", run, **autotune.knobs(C.FORM_LANE_SETS))
    assert {(t["tile_w"], t["tile_h"]) for t in seen} >= set(autotune.SHAPES)


def test_forms_by_size():
    """The form that measured ahead of the lane sets, or these, at each of the sizes
    beside the rule."""
    for n, W, H, k, want, *K in [
        (1_400_000, 162, 93, 5, C.FORM_ROW_WAVES),
        (50_000, 203, 152, 11, C.FORM_ROW_WAVES),
        # few candidates, ordinary and many on small images
        (26_667, 400, 300, 3, C.FORM_LANE_SETS),
        (48_000, 400, 300, 5, C.FORM_ROW_TILES),
        (263_000, 355, 357, 5, C.FORM_ROW_WAVES),
        (2_120_000, 1448, 1449, 5, C.FORM_ROW_TILES),
        (148_640, 963, 964, 5, C.FORM_LANE_SETS),
        (100_500, 781, 585, 7, C.FORM_LANE_SETS),
        (152_300, 781, 585, 7, C.FORM_ROW_TILES),
        # and of rows of many neighbours
        (135_720, 386, 292, 7, C.FORM_ROW_TILES, 32),
        (614_280, 621, 350, 7, C.FORM_ROW_TILES, 32),
        (614_280, 621, 350, 7, C.FORM_ROW_WAVES, 16),
        # wide windows
        (58_765, 400, 340, 9, C.FORM_LANE_SETS),
        (133_926, 500, 503, 13, C.FORM_LANE_SETS),
        (150_000, 500, 503, 9, C.FORM_LANE_SETS),
        (682_666, 640, 480, 15, C.FORM_LANE_SETS),
        (3_602_000, 345, 261, 9, C.FORM_ROW_WAVES),
        (1_896_000, 640, 480, 9, C.FORM_ROW_WAVES),
        (1_614_000, 683, 685, 9, C.FORM_LANE_SETS),
        (1_860_000, 516, 519, 9, C.FORM_LANE_SETS, 32),
        (398_222, 1280, 720, 9, C.FORM_ROW_TILES),
        (20_000_000, 1920, 1080, 15, C.FORM_ROW_TILES),
    ]:
        K = K[0] if K else 8
        assert form(n, W, H, kernel_size=k, num_point_cloud_per_sp=K) == want, (n, W, H, k, K)


def test_clouds_whose_rows_a_tile_cannot_count():
    """The tiles add the points of k + 3 rows in 31 bits, and rows of a caller's table
    may share their buckets."""
    for k in (5, 8, 9, 16):
        most = (2**31 - 1) // (k + 3)
        assert form(most, 8000, 8000, kernel_size=k) == C.FORM_ROW_TILES
        assert form(most + 1, 8000, 8000, kernel_size=k) == C.FORM_ROW_WAVES


def test_lists_whose_windows_cover_the_view():
    """Lists for which the cones' pass pays take the lane sets, where a workspace
    holds the cones."""
    full = lambda W, H: C._lib.epcq_sampling_workspace_size(300_000, H, W)  # noqa: E731
    for R, W, H, k, want in [
        (4096, 800, 800, 5, C.FORM_ROW_WAVES),
        (25_599, 200, 200, 5, C.FORM_ROW_WAVES),
        (25_600, 200, 200, 5, C.FORM_LANE_SETS),
        (35_208, 216, 163, 11, C.FORM_LANE_SETS),
        # windows of more than 12 columns: where the cones are made at all
        (288, 512, 508, 15, C.FORM_ROW_WAVES),  # 4 * 225 * 289 buckets >= 512 * 508
        (289, 512, 508, 15, C.FORM_LANE_SETS),
        (2076, 551, 551, 15, C.FORM_ROW_WAVES),
        (2076, 551, 475, 15, C.FORM_LANE_SETS),
        (2076, 551, 475, 12, C.FORM_ROW_WAVES),
    ]:
        assert form(300_000, W, H, rays=R, kernel_size=k) == want, (R, W, H, k)
        for ws in (0, W * H * 24 - 1):
            assert ws < full(W, H)
            assert form(300_000, W, H, rays=R, kernel_size=k, ws=ws) == C.FORM_ROW_WAVES, (R, W, H, k)
