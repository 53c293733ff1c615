"""The batched kernels' launch configuration: what a fresh context has, and
what a call that leaves the shape alone keeps."""
import time

import pytest

from patchmatch_amd import synth
from patchmatch_amd._lib import Context, Keyframe
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
