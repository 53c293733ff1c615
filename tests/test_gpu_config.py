"""The batched kernels' launch configuration: what a fresh context has, and
what a call that leaves the shape alone keeps."""
import time

import numpy as np
import pytest

from oracle import or_py
from patchmatch_amd import synth
from patchmatch_amd._lib import PMP_MAPS_INIT, PMP_MAPS_WORK, Context, Keyframe
from patchmatch_amd.params import config1_params

pytestmark = pytest.mark.gpu


def test_default_shape_is_kept():
    with Context(0) as ctx:
        fresh = ctx.batch_get_config()
        ctx.batch_set_config(use_graph=0)   # a caller who only wants direct launches
        assert ctx.batch_get_config() == dict(fresh, use_graph=0)
        ctx.batch_set_config()
        assert ctx.batch_get_config() == fresh


def test_one_band_keeps_pace():
    """xcd_bands 0 (every block takes its tiles from one list) is not slower than
    by half: its blocks all contend for the same heads.  It took ten times as
    long where a compare-and-swap handed the tiles out."""
    kf = synth.make_keyframe(5, 960, 480, 1, baseline=(0.05, 0.4), spheres=4)
    p = config1_params(iterations=4)
    ms = {}
    with Context(0) as ctx:
        ctx.image_put(1, kf.ref)
        ctx.image_put(2, kf.views[0])
        kfs = [Keyframe.make(1, kf.ref_pose, [2], kf.view_poses)] * 8
        for bands in (1, 0, 1, 0):
            ctx.batch_set_config(xcd_bands=bands)
            t = []
            for _ in range(4):
                t0 = time.perf_counter()
                ctx.batch_densify(p, kfs)
                ctx.synchronize()
                t.append(time.perf_counter() - t0)
            ms[bands] = min(ms.get(bands, 1e9), 1e3 * min(t))
            print(f"[config] xcd_bands {bands}: {min(t) * 1e3:.2f} ms", flush=True)
    assert ms[0] < 1.5 * ms[1], ms


@pytest.mark.parametrize("views,rows", [((1,) * 7 + (4,), 4), ((4,) + (2,) * 7, 4), ((2,) * 4 + (4,) * 4, 8),
                                        ((3,) * 7 + (4,), 8), ((1, 1, 3, 3, 3, 3, 3, 3), 4)])
def test_mixed_view_counts(views, rows):
    """A batch takes the form that most of its work is better with: tiles of 4
    rows where one or two views dominate, of 8 otherwise."""
    W, H = 420, 290
    kf = synth.make_keyframe(6, W, H, 4, baseline=(0.05, 0.4), spheres=4)
    p = config1_params(iterations=1)
    with Context(0) as ctx:
        ctx.image_put(1, kf.ref)
        for v, img in enumerate(kf.views):
            ctx.image_put(2 + v, img)
        kfs = [Keyframe.make(1, kf.ref_pose, [2 + v for v in range(n)], kf.view_poses[:n]) for n in views]
        ctx.debug_epochs(1)
        ctx.batch_densify(p, kfs)
        rep = ctx.debug_epoch_report()
        got = [ctx.batch_get_maps(k, (H, W)) for k in range(len(kfs))]
        ctx.debug_epochs(0)
        assert rep["tiles"] == 8 * -(-((W + 1) // 2) // 32) * -(-H // (2 * rows)) and rep["violations"] == 0, rep
        for k, n in enumerate(views):   # the same bits as alone
            ctx.set_views(1, kf.ref_pose, [2 + v for v in range(n)], kf.view_poses[:n])
            ctx.densify(p)
            for a, b in zip(ctx.get_maps(2), got[k]):
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (k, n)


# (W, H, views, keyframes, tile_rows, blocks_per_cu): whether the passes of a call share a launch on 256 CUs
@pytest.mark.parametrize("W,H,n,count,rows,bpc,one", [
    (203, 97, 1, 1, 4, 3, 0), (640, 320, 2, 1, 2, 1, 1), (640, 320, 2, 1, 2, 2, 1), (701, 187, 3, 1, 2, 1, 1),
    (960, 480, 1, 9, 2, 0, 1), (960, 480, 4, 35, 2, 0, 1),     # 10.5 and 30.8 tiles to a block
])
def test_passes_share_a_launch(W, H, n, count, rows, bpc, one):
    kf = synth.make_keyframe(7, W, H, 4, baseline=(0.05, 0.4), spheres=4)
    p = config1_params(iterations=2)
    with Context(0) as ctx:
        ctx.image_put(1, kf.ref)
        for v, img in enumerate(kf.views):
            ctx.image_put(2 + v, img)
        k = Keyframe.make(1, kf.ref_pose, [2 + v for v in range(n)], kf.view_poses[:n])
        ctx.batch_set_config(tile_rows=rows, blocks_per_cu=bpc)
        ctx.batch_densify(p, [k] * count)
        shape = ctx.debug_launch()
        got = [ctx.batch_get_maps(k, (H, W)) for k in {0, count // 2, count - 1}]
        assert shape["one_launch"] == one, shape
        ctx.set_views(1, kf.ref_pose, [2 + v for v in range(n)], kf.view_poses[:n])
        ctx.densify(p)
        want = ctx.get_maps(2)
        for g in got:
            assert all(np.array_equal(a.view(np.uint32), b.view(np.uint32)) for a, b in zip(g, want))


# lanes and quads on both sides of the lines between them (on 256 CUs), sizes that do not fill their tiles
@pytest.mark.parametrize("W,H,n,edge", [(601, 303, 1, 0), (601, 303, 2, 2), (601, 303, 5, 1), (601, 303, 4, 0),
                                        (801, 410, 3, 2), (801, 410, 5, 0), (961, 470, 2, 0), (961, 470, 1, 2)])
def test_initial_scores(W, H, n, edge):
    """Initial planes and scores by the form that the launch takes, against the oracle bit for bit."""
    kf = synth.make_keyframe(8, W, H, n, baseline=(0.05, 0.4), spheres=4)
    p = config1_params(iterations=0, seed=4, topk=min(n, 2), edge_mode=edge)
    want = or_py.densify(or_py.Keyframe.from_synth(kf), p, None)
    with Context(0) as ctx:
        ctx.load_keyframe(kf.ref, kf.views, kf.ref_pose, kf.view_poses)
        ctx.densify(p)
        got = ctx.get_maps(2)
        for name, g, o in (("plane", got[0][..., :3], want["plane"]), ("depth", got[1], want["depth"]),
                           ("score", got[2], want["score"])):
            eq = np.ascontiguousarray(g).view(np.uint32) == np.ascontiguousarray(o).view(np.uint32)
            assert eq.all(), f"{name}: {np.count_nonzero(~eq)} of {eq.size} differ"
        # the score call takes the same form
        ctx.random_initialization(p)
        plane, depth, score = ctx.get_maps(PMP_MAPS_INIT)
        ctx.set_maps(plane, depth, np.full_like(score, 7.0))
        ctx.score_plane_depth(p)
        again = ctx.get_maps(PMP_MAPS_WORK)[2]
        scored = again != 7.0
        assert scored.any() and np.array_equal(again[scored].view(np.uint32), score[scored].view(np.uint32))


@pytest.mark.parametrize("n", [5, 6, 10])   # groups of 3 + 2, 3 + 3 and 4 + 3 + 3 views
def test_several_groups_in_one_launch(n):
    """Quads with more than one group of views, all passes in one launch: the
    oracle's maps for every keyframe of the batch, bit for bit."""
    W, H = 403, 291
    kf = synth.make_keyframe(9, W, H, n, baseline=(0.05, 0.4), spheres=4)
    p = config1_params(iterations=2, seed=n)
    want = or_py.densify(or_py.Keyframe.from_synth(kf), p, kf.mask)
    with Context(0) as ctx:
        ctx.image_put(1, kf.ref)
        ctx.image_put(90, kf.mask)
        for v, img in enumerate(kf.views):
            ctx.image_put(2 + v, img)
        k = Keyframe.make(1, kf.ref_pose, [2 + v for v in range(n)], kf.view_poses, mask_id=90)
        for _ in range(2):   # the graph's first launch and a replay
            ctx.batch_densify(p, [k] * 9)
            shape = ctx.debug_launch()
            assert (shape["form"], shape["tile_rows"], shape["one_launch"]) == (1, 8, 1), shape
            for i in range(9):
                got = ctx.batch_get_maps(i, (H, W))
                for name, g, o in (("plane", got[0][..., :3], want["plane"]), ("depth", got[1], want["depth"]),
                                   ("score", got[2], want["score"])):
                    eq = np.ascontiguousarray(g).view(np.uint32) == np.ascontiguousarray(o).view(np.uint32)
                    assert eq.all(), f"keyframe {i} {name}: {np.count_nonzero(~eq)} of {eq.size} differ"
