"""Copies that share a context's state or lie on the other side of a line of the
staged copies: a server whose images and results move on several threads at
once, and the pruner's read-back in sizes below and above the one from which it
takes the copying threads."""
import threading

import numpy as np
import pytest

from patchmatch_amd import synth
from patchmatch_amd._lib import Server
from patchmatch_amd.params import config1_params

pytestmark = pytest.mark.gpu


def test_server_threads(gpu_ctx):
    """Two threads submit keyframes whose images are above 6 MiB, the third
    fetches: the maps of the one-keyframe path, bit for bit."""
    W, H, n = 3600, 1820, 3
    p = config1_params(iterations=1)
    seqs = [synth.sequence_gpu(40 + k, 2, W, H, with_gt=False) for k in range(2)]
    want = []
    for seq in seqs:
        gpu_ctx.load_keyframe(seq["images"][0], seq["images"][1:], seq["poses"][0], seq["poses"][1:])
        gpu_ctx.densify(p)
        want.append(gpu_ctx.get_maps(2))
    srv = Server(0, max_slots=2)
    tickets, errors = [], []
    ready = threading.Semaphore(0)

    def submit(k):
        try:
            seq = seqs[k]
            for r in range(n):
                base = 1000 * k + 10 * r   # images of their own: every request uploads
                tickets.append((k, srv.submit(p, base, seq["poses"][0], [base + 1], seq["poses"][1:], (H, W),
                                              ref=seq["images"][0], views=seq["images"][1:])))
                ready.release()
        except Exception as e:   # shown by the main thread
            errors.append(e)
            ready.release()

    ts = [threading.Thread(target=submit, args=(k,)) for k in range(2)]
    print(f"[copy] server, {2 * n} requests of {W}x{H} on two threads", flush=True)
    for t in ts:
        t.start()
    for done in range(2 * n):
        ready.acquire()
        assert not errors, errors
        k, ticket = tickets[done]
        srv.wait(ticket)
        got = srv.fetch(ticket)[:4]
        for a, b in zip(got, want[k]):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (k, done)
    for t in ts:
        t.join()
    srv.close()


@pytest.mark.parametrize("W,H", [(320, 160), (1098, 494), (1363, 677)])   # points and map: 2, 21 and 36 MB
def test_pruner_read_back(gpu_ctx, W, H):
    rng = np.random.default_rng(W)
    d = rng.random((H, W), dtype=np.float32) + 1.0
    bgr = rng.integers(0, 256, (H, W, 3), dtype=np.uint8)
    pose = np.concatenate([np.eye(3).ravel(), np.zeros(3)])
    gpu_ctx.pruner_reset()
    gpu_ctx.pruner_add_view(d, pose, bgr)
    pruned, pts, cols, kps = gpu_ctx.pruner_prune(0.01, (H, W))
    gpu_ctx.pruner_reset()
    assert np.array_equal(pruned, d)          # a single view: nothing prunes it
    assert len(pts) == W * H
    rows, columns = kps[:, 0], kps[:, 1]
    assert np.array_equal(rows * W + columns, np.arange(W * H))
    assert np.array_equal(cols, bgr.reshape(-1, 3))
    B = synth.bearings(W, H).reshape(-1, 3)
    # bearings to float32's rounding at worst, depths below 2
    assert np.abs(pts - d.reshape(-1, 1).astype(np.float64) * B).max() < 1e-6
