"""The red-black passes of a call run in one launch or in one launch each,
depending on the number of tiles and of blocks in flight: both forms, at odd
sizes, with one tile per block, many, and a band that holds fewer tiles than
there are blocks, against the oracle bit for bit; the same maps again when the
graph is replayed, and for a batch whose bands hold several keyframes."""
import numpy as np
import pytest

from conftest import cached
from oracle import or_py
from patchmatch_amd import synth
from patchmatch_amd._lib import Keyframe
from patchmatch_amd.params import EDGE_ZERO, config1_params, default_params

pytestmark = pytest.mark.gpu


def _same(got, want, tag):
    for name, g, o in (("plane", got[0][..., :3], want["plane"]), ("depth", got[1], want["depth"]),
                       ("score", got[2], want["score"])):
        eq = np.ascontiguousarray(g).view(np.uint32) == np.ascontiguousarray(o).view(np.uint32)
        assert eq.all(), f"{tag} {name}: {np.count_nonzero(~eq)} of {eq.size} differ"


def _kf(W, H, n):
    return cached(f"passes_{W}x{H}_{n}", lambda: synth.make_keyframe(31 + n, W, H, n, baseline=(0.05, 0.4), spheres=6))


def _oracle(kf, p, tag):
    return cached(f"passes_oracle_{tag}", lambda: or_py.densify(or_py.Keyframe.from_synth(kf), p, kf.mask))


# tiles of the four: 28, 800, 800, 516
@pytest.mark.parametrize("W,H,n,rows,bpc", [(203, 97, 1, 4, 3), (640, 320, 2, 2, 1), (640, 320, 2, 2, 2),
                                            (701, 187, 3, 2, 1)])
def test_launch_forms_bitwise(gpu_ctx, W, H, n, rows, bpc):
    kf = _kf(W, H, n)
    p = config1_params(iterations=3, seed=40 + n, edge_mode=EDGE_ZERO if n == 3 else 0)
    want = _oracle(kf, p, f"{W}x{H}_{n}")
    cfg = gpu_ctx.batch_get_config()
    gpu_ctx.load_keyframe(kf.ref, kf.views, kf.ref_pose, kf.view_poses)
    try:
        gpu_ctx.batch_set_config(tile_rows=rows, blocks_per_cu=bpc, use_graph=1, xcd_bands=1)
        print(f"[passes] {W}x{H}, {n} views, tile_rows {rows}, {bpc} blocks per CU", flush=True)
        for k in range(3):   # the graph's first launch and two replays
            gpu_ctx.densify(p, kf.mask)
            _same(gpu_ctx.get_maps(2), want, f"run {k}")
        gpu_ctx.batch_set_config(tile_rows=rows, blocks_per_cu=bpc, use_graph=0, xcd_bands=0)
        gpu_ctx.densify(p, kf.mask)
        _same(gpu_ctx.get_maps(2), want, "one band")
    finally:
        gpu_ctx.batch_set_config(**cfg)


def test_batch_bands_over_keyframes(gpu_ctx):
    """Bands that hold whole small keyframes and parts of larger ones."""
    p = default_params(iterations=2, seed=77)
    shapes = [(203, 97, 1), (640, 320, 2), (203, 97, 1), (701, 187, 3)]
    kfs = [_kf(*s) for s in shapes]
    descs = []
    for k, kf in enumerate(kfs):
        base = 7000 + 100 * k
        gpu_ctx.image_put(base, kf.ref)
        gpu_ctx.image_put(base + 50, kf.mask)
        for v, img in enumerate(kf.views):
            gpu_ctx.image_put(base + 1 + v, img)
        descs.append(Keyframe.make(base, kf.ref_pose, [base + 1 + v for v in range(len(kf.views))], kf.view_poses,
                                   mask_id=base + 50))
    cfg = gpu_ctx.batch_get_config()
    try:
        for bpc in (1, 4):
            gpu_ctx.batch_set_config(tile_rows=2, blocks_per_cu=bpc, use_graph=1, xcd_bands=1)
            print(f"[passes] batch of 4, {bpc} blocks per CU", flush=True)
            gpu_ctx.batch_densify(p, descs)
            for k, kf in enumerate(kfs):
                want = _oracle(kf, p, f"batch_{shapes[k][0]}")
                _same(gpu_ctx.batch_get_maps(k, (kf.H, kf.W)), want, f"keyframe {k}, {bpc} blocks per CU")
    finally:
        gpu_ctx.batch_set_config(**cfg)
