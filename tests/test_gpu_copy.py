"""Copies between host memory and the device at the edges of their chunks: one
that the caller copies alone, several pieces, whole chunks, more chunks than
the ring holds, rows with a pitch, maps in one transfer, pinned memory (which
goes straight), and contexts on several threads at once; whole numbers, so the
bytes have to be the same."""
import ctypes
import threading

import numpy as np
import pytest
import torch

from patchmatch_amd._lib import Context, PMP_MAPS_WORK

pytestmark = pytest.mark.gpu


# the caller alone; just above that; less than a chunk; 4.5 chunks (the ring holds 2), with and without a pitch; 12 chunks
@pytest.mark.parametrize("W,H,pitch", [(511, 1024, 511), (801, 1000, 900), (2047, 1024, 2047), (2049, 1024, 2049),
                                       (4099, 4613, 4099), (4099, 4613, 5003), (8192, 6144, 8192)])
def test_images_round_trip(gpu_ctx, W, H, pitch):
    rng = np.random.default_rng(W + pitch)
    full = rng.integers(0, 256, (H, pitch), dtype=np.uint8)
    print(f"[copy] {W}x{H}, pitch {pitch}", flush=True)
    for k in range(2):
        img = full if k == 0 else full[::-1].copy()
        # pitched rows: the call itself, as the wrapper passes contiguous images only
        gpu_ctx._chk(gpu_ctx.L.pmp_image_put(gpu_ctx.h, 900 + k, img.ctypes.data_as(ctypes.POINTER(ctypes.c_uint8)),
                                             W, H, pitch, 0), "pmp_image_put")
    for k in range(2):
        assert np.array_equal(gpu_ctx.image_get(900 + k, (H, W)), full[:, :W] if k == 0 else full[::-1, :W])
        gpu_ctx.image_drop(900 + k)


def _maps_round_trip(ctx, W, H, seed, out):
    rng = np.random.default_rng(seed)
    img = rng.integers(0, 256, (H, W), dtype=np.uint8)
    pose = np.concatenate([np.eye(3).ravel(), np.zeros(3)])
    for k in range(2):
        ctx.image_put(10 + k, img)
    ctx.set_views(10, pose, [11], [pose + np.r_[np.zeros(9), 0.1, 0, 0]])
    for _ in range(3):
        maps = [rng.random(s, dtype=np.float32) for s in ((H, W, 4), (H, W), (H, W))]
        ctx.set_maps(*maps)
        got = ctx.get_maps(PMP_MAPS_WORK)
        out.append(all(np.array_equal(a.view(np.uint32), b.view(np.uint32)) for a, b in zip(got, maps)))


@pytest.mark.parametrize("W,H", [(96, 64), (640, 321), (1363, 677)])
def test_maps_from_several_threads(W, H):
    ctxs = [Context(0) for _ in range(3)]
    outs = [[] for _ in ctxs]
    print(f"[copy] maps {W}x{H} on three threads", flush=True)
    ts = [threading.Thread(target=_maps_round_trip, args=(c, W, H, k, o)) for k, (c, o) in enumerate(zip(ctxs, outs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for c in ctxs:
        c.close()
    assert [o for o in outs] == [[True] * 3] * 3


def test_pinned_memory(gpu_ctx):
    img = torch.empty((1024, 3000), dtype=torch.uint8, pin_memory=True).random_(0, 256)
    gpu_ctx.image_put(910, img.numpy())
    assert np.array_equal(gpu_ctx.image_get(910, (1024, 3000)), img.numpy())
    gpu_ctx.image_drop(910)
