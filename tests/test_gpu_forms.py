"""The propagation evaluates planes one per lane, by quads of lanes, or by
quads with four times the waves to a tile, depending on the pixels and views of
a launch (and on an explicit tile size): each form against the oracle bit for
bit, with view counts that split into the quads' groups in every way, tap
counts that are and are not multiples of four, every aggregation and edge mode,
sizes that do not fill their tiles, and on both sides of the sizes where the
form changes."""
import numpy as np
import pytest

from conftest import cached
from oracle import or_py
from patchmatch_amd import synth
from patchmatch_amd._lib import PMP_MAPS_INIT, PMP_MAPS_WORK
from patchmatch_amd.params import (AGG_FOLD_INDEP, AGG_MAX, AGG_REF_FOLD, AGG_TOPK_MEAN, EDGE_CLAMP, EDGE_WRAP,
                                   EDGE_ZERO, config1_params)

pytestmark = pytest.mark.gpu

# W, H, views, half, stride, aggregation, edge; tile_rows asked for (0: default), tile rows expected
CASES = [
    (203, 97, 1, 3, 1, AGG_REF_FOLD, EDGE_WRAP, 0, 2),
    (130, 66, 2, 3, 3, AGG_TOPK_MEAN, EDGE_ZERO, 0, 2),
    (203, 97, 3, 7, 3, AGG_MAX, EDGE_CLAMP, 0, 2),
    (203, 97, 4, 5, 2, AGG_FOLD_INDEP, EDGE_ZERO, 4, 4),
    (97, 130, 5, 4, 2, AGG_REF_FOLD, EDGE_WRAP, 0, 2),
    (203, 97, 6, 3, 1, AGG_TOPK_MEAN, EDGE_ZERO, 8, 8),
    (203, 97, 7, 5, 2, AGG_REF_FOLD, EDGE_CLAMP, 8, 8),
    (65, 48, 9, 3, 2, AGG_FOLD_INDEP, EDGE_WRAP, 8, 8),
    (203, 97, 10, 5, 1, AGG_REF_FOLD, EDGE_ZERO, 0, 2),
    (403, 203, 5, 3, 1, AGG_MAX, EDGE_WRAP, 0, 2),
    (640, 305, 1, 3, 2, AGG_REF_FOLD, EDGE_WRAP, 0, 2),      # just below and above one view's change
    (640, 308, 1, 3, 2, AGG_TOPK_MEAN, EDGE_ZERO, 0, 4),
    (903, 450, 2, 3, 3, AGG_MAX, EDGE_WRAP, 8, 8),
    (903, 450, 3, 3, 2, AGG_REF_FOLD, EDGE_ZERO, 2, 2),
    (1363, 691, 4, 3, 3, AGG_TOPK_MEAN, EDGE_CLAMP, 0, 8),
    (1363, 691, 3, 3, 3, AGG_REF_FOLD, EDGE_WRAP, 4, 4),
]


@pytest.mark.parametrize("W,H,n,half,stride,agg,edge,rows,want_rows", CASES)
def test_forms_bitwise(gpu_ctx, W, H, n, half, stride, agg, edge, rows, want_rows):
    kf = cached(f"forms_{W}x{H}_{n}", lambda: synth.make_keyframe(50 + n, W, H, n, baseline=(0.05, 0.4), spheres=5))
    p = config1_params(iterations=2 if W < 600 else 1, seed=60 + n, patch_half=half, patch_stride=stride,
                       agg_mode=agg, topk=min(n, 3), edge_mode=edge)
    want = cached(f"forms_oracle_{W}x{H}_{n}_{half}_{stride}_{agg}_{edge}",
                  lambda: or_py.densify(or_py.Keyframe.from_synth(kf), p, kf.mask))
    cfg = gpu_ctx.batch_get_config()
    gpu_ctx.load_keyframe(kf.ref, kf.views, kf.ref_pose, kf.view_poses)
    print(f"[forms] {W}x{H}, {n} views, patch {half}/{stride}, tile_rows {rows}", flush=True)
    try:
        # tile_rows 2 with 0 blocks per CU is the default, which chooses the rows itself
        gpu_ctx.batch_set_config(tile_rows=rows or 2, blocks_per_cu=4 if rows else 0, use_graph=1, xcd_bands=1)
        gpu_ctx.debug_epochs(1)
        gpu_ctx.densify(p, kf.mask)
        rep = gpu_ctx.debug_epoch_report()
        got = gpu_ctx.get_maps(2)
    finally:
        gpu_ctx.debug_epochs(0)
        gpu_ctx.batch_set_config(**cfg)
    assert rep["tiles"] == -(-((W + 1) // 2) // 32) * -(-H // (2 * want_rows)) and rep["violations"] == 0, rep
    for name, g, o in (("plane", got[0][..., :3], want["plane"]), ("depth", got[1], want["depth"]),
                       ("score", got[2], want["score"])):
        eq = np.ascontiguousarray(g).view(np.uint32) == np.ascontiguousarray(o).view(np.uint32)
        assert eq.all(), f"{name}: {np.count_nonzero(~eq)} of {eq.size} differ"


# init tiles: 100, 357, 770 (16, 32 and 64 pixels to a wave on 256 CUs)
@pytest.mark.parametrize("W,H,n", [(203, 97, 7), (403, 203, 5), (640, 305, 2)])
def test_score_forms_bitwise(gpu_ctx, W, H, n):
    """Scores of the initial planes by the score call: those of the initialisation."""
    kf = cached(f"forms_{W}x{H}_{n}", lambda: synth.make_keyframe(50 + n, W, H, n, baseline=(0.05, 0.4), spheres=5))
    p = config1_params(seed=3, edge_mode=EDGE_ZERO if n == 5 else EDGE_WRAP)
    gpu_ctx.load_keyframe(kf.ref, kf.views, kf.ref_pose, kf.view_poses)
    print(f"[forms] score {W}x{H}, {n} views", flush=True)
    gpu_ctx.random_initialization(p)
    plane, depth, score = gpu_ctx.get_maps(PMP_MAPS_INIT)
    gpu_ctx.set_maps(plane, depth, np.full_like(score, 7.0))
    gpu_ctx.score_plane_depth(p)
    got = gpu_ctx.get_maps(PMP_MAPS_WORK)[2]
    scored = got != 7.0
    h = p.patch_half + 1
    assert scored[h + 1:H - h, h + 1:W - h].all() and not scored[0].any()
    assert np.array_equal(got[scored].view(np.uint32), score[scored].view(np.uint32))
    assert np.abs(got[scored]).max() <= 1.0 and np.ptp(got[scored]) > 0.5
