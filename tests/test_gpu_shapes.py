"""Read-backs into a shape that the caller names: what the map does not fill is 0."""
import numpy as np
import pytest

from patchmatch_amd import synth
from patchmatch_amd._lib import Keyframe
from patchmatch_amd.params import config1_params

pytestmark = pytest.mark.gpu


def _used_memory(shape):
    """Leaves freed memory of the size behind that is not 0."""
    for _ in range(4):
        np.full(shape, np.nan, np.float32)


def test_pruner_map_in_a_larger_array(gpu_ctx):
    W, H = 64, 32
    d = np.random.default_rng(1).random((H, W), dtype=np.float32) + 1.0
    pose = np.concatenate([np.eye(3).ravel(), np.zeros(3)])
    gpu_ctx.pruner_reset()
    gpu_ctx.pruner_add_view(d, pose, np.zeros((H, W, 3), np.uint8))
    _used_memory((2 * H, W))
    got = gpu_ctx.pruner_get_map(0, (2 * H, W))
    gpu_ctx.pruner_reset()
    assert np.array_equal(got[:H], d) and not got[H:].any()


def test_batch_maps_in_larger_arrays(gpu_ctx):
    W, H = 96, 48
    kf = synth.make_keyframe(3, W, H, 1, baseline=(0.05, 0.4), spheres=2)
    gpu_ctx.image_put(8800, kf.ref)
    gpu_ctx.image_put(8801, kf.views[0])
    gpu_ctx.batch_densify(config1_params(iterations=1),
                          [Keyframe.make(8800, kf.ref_pose, [8801], kf.view_poses)])
    want = gpu_ctx.batch_get_maps(0, (H, W))
    _used_memory((2 * H, W, 4))
    _used_memory((2 * H, W))
    got = gpu_ctx.batch_get_maps(0, (2 * H, W))
    for a, b in zip(got, want):
        assert np.array_equal(a[:H].view(np.uint32), b.view(np.uint32)) and not a[H:].any()
