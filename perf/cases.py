"""What is measured of the densifier: cases of the work its users have it do.

Every case goes through the public Python classes (``Context``, ``Server``) as
a program does that feeds the densify thread's keyframes to the library and
takes the maps back to the host.  A case's fields:

kind      what a pass is:
  densify    one keyframe: select it, densify, read the final maps back;
  warm       one keyframe of the densify thread at its own loop: random
             initialisation, landmark seeding (``landmarks`` points), the
             previous result warped in, the red-black passes, copy-back and
             post-processing, read-back;
  batch      ``count`` keyframes of mixed sizes in one call, all maps read back;
  served     ``count`` requests submitted to a server at once, then fetched;
  score      the scores and unit normals of a given plane map;
  clean      the geometric-consistency filter over a window of ``views`` depth maps;
  fuse       the point fusion's window of ``views`` cleaned maps: filled, the
             head pruned, the points read back;
  thumbnail  one camera frame to the pooled grey thumbnail, and that read back.
W, H      keyframe size (largest of a batch; the thumbnail's for ``thumbnail``)
views     neighbours of a keyframe, or maps of a window
base      the parameter set (``params.CONFIGS``); the other fields override it

Scenes are the seeded synthetic room of the repository's own workloads,
rendered on the GPU, textured to the working resolution.
"""
import math

import numpy as np
import torch

from patchmatch_amd import params as pm
from patchmatch_amd import synth
from patchmatch_amd._lib import PMP_MAPS_FINAL, PMP_MAPS_WORK, Context, Keyframe, Server

PARAM_FIELDS = ("patch_half", "patch_stride", "iterations", "n_refine", "topk")
ENUM_FIELDS = ("agg_mode", "edge_mode", "coverage_mode", "init_mode")
CHANNELS = 3        # of a camera frame
MIN_CONSISTENT = 3  # the densify thread's own setting


def listed():
    return [
        # the smallest keyframe: 480x240, two neighbours, dense 7x7 patch; the launches weigh most here
        dict(name="densify_480x240_2v", kind="densify", W=480, H=240, views=2, base="config0"),
        # the densify thread's loop at the example configuration (640x320, 2 neighbours, 4 iterations,
        # the reference's constants), landmarks and the previous result included
        dict(name="warm_640x320_2v", kind="warm", W=640, H=320, views=2, base="default", iterations=4, landmarks=1500),
        # the headline: 1920x960, 6 neighbours, best 3 of 6, 8 iterations
        dict(name="densify_1920x960_6v", kind="densify", W=1920, H=960, views=6, base="config1"),
        # the same keyframe in a running trajectory: 2 iterations from the previous result
        dict(name="warm_1920x960_6v", kind="warm", W=1920, H=960, views=6, base="config1", iterations=2, landmarks=0),
        # odd sizes, zero edges, the best view's score, a dense small patch
        dict(name="densify_1363x677_4v_zero", kind="densify", W=1363, H=677, views=4, base="config1", iterations=4,
             agg_mode="max", edge_mode="zero", patch_half=3, patch_stride=1),
        # the largest keyframe: 2880x1440, 10 neighbours
        dict(name="densify_2880x1440_10v", kind="densify", W=2880, H=1440, views=10, base="config1"),
        # a backlog of keyframes of mixed sizes and view counts in one call
        dict(name="batch_8", kind="batch", W=1920, H=960, views=6, base="config1", iterations=4, count=8),
        # a stream of small requests served together
        dict(name="served_6", kind="served", W=960, H=480, views=4, base="config1", iterations=4, count=6),
        # scores and normals of a given plane map (a map from elsewhere is checked against the images)
        dict(name="score_960x480_6v", kind="score", W=960, H=480, views=6, base="config1"),
        # the densify thread's 5-deep consistency window
        dict(name="clean_1920x960_5", kind="clean", W=1920, H=960, views=5, base="config1"),
        # the point-cloud thread's 5-deep window
        dict(name="fuse_1920x960_5", kind="fuse", W=1920, H=960, views=5, base="config1"),
        # a full camera frame to its keyframe's thumbnail
        dict(name="thumbnail_5760x2880", kind="thumbnail", W=1920, H=960, views=0, base="config1", frame_W=5760,
             frame_H=2880),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["densify", "densify", "densify", "warm", "warm", "batch", "served", "score", "clean", "fuse",
                       "thumbnail"])
    W = _log_int(rng, 320, 2880 if kind == "densify" else 1920)
    H = max(96, W // 2 + rng.randint(-W // 16, W // 16))
    c = dict(kind=kind, W=W, H=H, views=rng.randint(1, 10), base="config1")
    if kind in ("densify", "warm", "batch", "served", "score"):
        c.update(agg_mode=rng.choice(["ref_fold", "max", "topk_mean", "topk_mean", "fold_indep"]),
                 edge_mode=rng.choice(["wrap", "wrap", "clamp", "zero"]), topk=rng.randint(1, 4),
                 coverage_mode=rng.choice(["full", "ref_grid"]), init_mode=rng.choice(["invdepth_hemi", "ref_uniform"]))
        half, stride = rng.choice([(5, 2), (5, 2), (3, 1), (4, 2), (7, 3), (5, 1)])
        c.update(patch_half=half, patch_stride=stride, iterations=rng.randint(1, 8 if kind == "densify" else 4))
    if kind == "warm":
        c.update(landmarks=rng.choice([0, 137, 1500, 6001]))
    if kind in ("batch", "served"):
        c.update(views=rng.randint(2, 6), count=rng.randint(2, 8))
    if kind == "score":
        c.update(W=min(W, 960), H=min(H, 480), agg_mode="topk_mean", coverage_mode="full")
    if kind in ("clean", "fuse"):
        c.update(views=rng.randint(3, 6))
    if kind == "thumbnail":
        f = rng.randint(1, 3)
        c.update(views=0, frame_W=W * f + rng.randint(0, 40), frame_H=H * f + rng.randint(0, 40))
    # no drawn case costs more than the largest listed one
    top = work(listed()[5])["flops"]
    while work(c)["flops"] > top:
        if c.get("iterations", 1) > 1:
            c["iterations"] -= 1
        else:
            c["views"] -= 1
    return c


def _params(case, seed):
    kw = {f: case[f] for f in PARAM_FIELDS if f in case}
    kw.update({f: pm.ENUMS[f][case[f]] for f in ENUM_FIELDS if f in case})
    return pm.CONFIGS[case["base"]](seed=seed, **kw)


def _taps(p):
    return (2 * p.patch_half // p.patch_stride + 1) ** 2


def _sizes(case):
    """The keyframe sizes and view counts of a batch or a request stream."""
    out = []
    for k in range(case["count"]):
        f = (1.0, 0.5, 0.73)[k % 3] if case["kind"] == "batch" else 1.0
        views = 2 + (case["views"] - 2 + 3 * k) % (case["views"] - 1)   # 2 to the case's, its own first
        out.append((max(160, int(case["W"] * f)), max(96, int(case["H"] * f)), views))
    return out


def work(case):
    p = _params(case, 0)
    px = case["W"] * case["H"]
    n, kind = case["views"], case["kind"]
    T = _taps(p)

    def densify(px, n):
        # per pixel and iteration the n_refine trials and, of the 8 propagation candidates, the fifth or so that
        # the penalty leaves a chance; once the initial plane
        ev = px * (1 + p.iterations * (p.n_refine + 1.6))
        return dict(bytes=px * (1 + n) + px * 28, flops=ev * (T * (19 + 52 * n) + 25 * n + 10))

    if kind in ("densify", "warm"):
        w = densify(px, n)
        if kind == "warm":
            w["flops"] += (px + case["landmarks"]) * (T * (19 + 52 * n) + 25 * n + 10)
            w["bytes"] += px * 20
        return w
    if kind in ("batch", "served"):
        parts = [densify(W * H, v) for W, H, v in _sizes(case)]
        return {k: sum(q[k] for q in parts) for k in ("bytes", "flops")}
    if kind == "score":
        return dict(bytes=px * (1 + n) + px * 32, flops=px * (T * (19 + 52 * n) + 25 * n + 10))
    if kind == "clean":
        return dict(bytes=px * 4 * (n + 1), flops=px * (n - 1) * 90.0)
    if kind == "fuse":
        return dict(bytes=px * (7 * n + 4 + 35), flops=px * (n - 1) * 90.0)
    fpx = case["frame_W"] * case["frame_H"]
    return dict(bytes=fpx * CHANNELS + px, flops=fpx * 6.0 + px * 9.0)


def _sequence(seed, n, W, H, with_gt=False):
    # texture scaled to the width: the finest octave stays about 3 px at 3 m
    return synth.sequence_gpu(seed, n, W, H, 0.2, with_gt=with_gt, base_freq=synth.TEX_FREQ_C1 * W / 1920.0)


def _nearest(k, n, count):
    return sorted((m for m in range(n) if m != k), key=lambda m: (abs(m - k), m))[:count]


def _landmarks(rng, poses, gt, n):
    """World points on the surfaces seen from poses, a few per cent off, as triangulated landmarks are."""
    H, W = gt.shape
    B = synth.bearings(W, H)
    r, c = rng.integers(0, H, n), rng.integers(0, W, n)
    X = (gt[r, c] * rng.normal(1.0, 0.02, n))[:, None] * B[r, c]
    return np.ascontiguousarray((X - poses[9:]) @ poses[:9].reshape(3, 3))


def _noisy_depths(rng, gts):
    """Depth maps as the densifier leaves them: close to the surface, a tenth of the pixels wrong, a tenth rejected."""
    out = []
    for g in gts:
        u = rng.random(g.shape, dtype=np.float32)
        d = g * (1.0 + 0.004 * (rng.random(g.shape, dtype=np.float32) - 0.5))
        d = np.where(u < 0.1, d * (0.5 + 10.0 * u), d)
        out.append(np.where(u > 0.9, 0.0, d).astype(np.float32))
    return out


def prepare(case, seed):
    kind, W, H, n = case["kind"], case["W"], case["H"], case["views"]
    rng = np.random.default_rng(seed)
    s = dict(case=case, p=_params(case, seed))
    if kind == "served":
        s["server"] = Server(0, max_slots=4, edge_mode=s["p"].edge_mode)
        seq = _sequence(seed, n + 4, W, H)
        s["seq"], s["refs"] = seq, [(1 + k % (n + 2), v) for k, (_, _, v) in enumerate(_sizes(case))]
        return s
    ctx = s["ctx"] = Context(0)
    if kind in ("densify", "warm"):
        m = n + (2 if kind == "warm" else 1)
        seq = _sequence(seed, m, W, H, with_gt=kind == "warm")
        for k in range(m):
            ctx.image_put(1 + k, seq["images"][k])
        ref = m // 2
        nb = _nearest(ref, m, n)
        s.update(mask=seq["mask"], ref=1 + ref, ref_pose=seq["poses"][ref], nb=[1 + k for k in nb],
                 nb_poses=[seq["poses"][k] for k in nb])
        if kind == "warm":
            # the previous keyframe's result, memorised as the densify thread does
            pb = _nearest(ref - 1, m, n)
            ctx.set_views(ref, seq["poses"][ref - 1], [1 + k for k in pb], [seq["poses"][k] for k in pb])
            ctx.densify(s["p"], s["mask"])
            ctx.memorize_result()
            s["xyz"] = _landmarks(rng, s["ref_pose"], seq["gt"][ref], case["landmarks"])
    elif kind == "batch":
        s["kfs"], s["shapes"] = [], []
        seqs = {}
        for k, (w, h, v) in enumerate(_sizes(case)):
            if (w, h) not in seqs:
                base = 100 * (1 + len(seqs))
                seqs[w, h] = base, _sequence(seed * 7 + len(seqs), n + 2, w, h)
                for m in range(n + 2):
                    ctx.image_put(base + m, seqs[w, h][1]["images"][m])
                ctx.image_put(base + 99, seqs[w, h][1]["mask"])
            base, seq = seqs[w, h]
            ref = k % (n + 2)
            nb = _nearest(ref, n + 2, v)
            s["kfs"].append(Keyframe.make(base + ref, seq["poses"][ref], [base + m for m in nb],
                                          [seq["poses"][m] for m in nb], mask_id=base + 99))
            s["shapes"].append((h, w))
    elif kind == "score":
        seq, plane, depth = _score_inputs(case, seed)
        for k in range(n + 1):
            ctx.image_put(1 + k, seq["images"][k])
        ctx.set_views(1, seq["poses"][0], [2 + k for k in range(n)], [seq["poses"][1 + k] for k in range(n)])
        ctx.set_maps(plane, depth, np.zeros((H, W), np.float32))
    elif kind in ("clean", "fuse"):
        s.update(_window(case, seed))
        if kind == "fuse":
            s["bgr"] = [np.ascontiguousarray(np.repeat(i[..., None], 3, -1)) for i in s["images"]]
    else:
        s["frame"] = _frame(case, rng)
    return s


def _frame(case, rng):
    g = rng.integers(0, 256, (case["frame_H"] // 8 + 2, case["frame_W"] // 8 + 2, CHANNELS), dtype=np.uint8)
    g = np.repeat(np.repeat(g, 8, 0), 8, 1)[:case["frame_H"], :case["frame_W"]]
    return np.ascontiguousarray(g ^ rng.integers(0, 16, (1, case["frame_W"], 1), dtype=np.uint8))


def _window(case, seed):
    """Depth maps, poses and images of a window of a trajectory, its centre first."""
    n = case["views"]
    seq = _sequence(seed, n, case["W"], case["H"], with_gt=True)
    order = [n // 2] + [k for k in range(n) if k != n // 2]
    d = _noisy_depths(np.random.default_rng(seed + 1), [seq["gt"][k] for k in order])
    return dict(depths=d, poses=[seq["poses"][k] for k in order], images=[seq["images"][k] for k in order])


def _score_inputs(case, seed):
    """The ground-truth planes of the first keyframe, half of them tilted."""
    seq = _sequence(seed, case["views"] + 1, case["W"], case["H"], with_gt=True)
    s_scene = synth._split_seeds(seed ^ 0x5E0, 2)[0]
    scene = synth.make_scene(s_scene, spheres=20, tube=True, cam_region=2.7,
                             base_freq=synth.TEX_FREQ_C1 * case["W"] / 1920.0)
    plane = synth.render_planes(scene, seq["poses"][0], case["W"], case["H"])
    plane = synth.tilt_planes(plane, np.random.default_rng(seed + 2), 0.5, 0.2)
    return seq, plane, seq["gt"][0].astype(np.float32)


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "served":
        srv, seq, shape = s["server"], s["seq"], (case["H"], case["W"])
        tickets = []
        for ref, v in s["refs"]:
            nb = _nearest(ref, len(seq["poses"]), v)
            tickets.append(srv.submit(s["p"], 1 + ref, seq["poses"][ref], [1 + m for m in nb],
                                      [seq["poses"][m] for m in nb], shape, ref=seq["images"][ref],
                                      views=[seq["images"][m] for m in nb], mask_id=1000, mask=seq["mask"]))
        out = []
        for t in tickets:
            srv.wait(t)
            out.append(srv.fetch(t)[:4])
        return out
    ctx = s["ctx"]
    if kind == "densify":
        ctx.set_views(s["ref"], s["ref_pose"], s["nb"], s["nb_poses"])
        ctx.densify(s["p"], s["mask"])
        return ctx.get_maps(PMP_MAPS_FINAL)
    if kind == "warm":
        ctx.set_views(s["ref"], s["ref_pose"], s["nb"], s["nb_poses"])
        ctx.random_initialization(s["p"])
        seeded = ctx.preinit_landmarks(s["p"], s["xyz"], s["mask"])
        warped = ctx.preinit_warp(s["p"], s["mask"])
        ctx.red_black_pass(s["p"], 0, s["p"].iterations)
        ctx.finalize(s["p"], s["mask"])
        return ctx.get_maps(PMP_MAPS_FINAL) + (seeded, warped)
    if kind == "batch":
        ctx.batch_densify(s["p"], s["kfs"])
        return [ctx.batch_get_maps(k, s["shapes"][k]) for k in range(len(s["kfs"]))]
    if kind == "score":
        ctx.score_plane_depth(s["p"])
        return {"score": ctx.get_maps(PMP_MAPS_WORK)[2], "normals": ctx.get_normals(PMP_MAPS_WORK)}
    if kind == "clean":
        return ctx.clean(s["depths"], s["poses"], 0.01, MIN_CONSISTENT)
    if kind == "fuse":
        ctx.pruner_reset()
        for d, pose, bgr in zip(s["depths"], s["poses"], s["bgr"]):
            ctx.pruner_add_view(d, pose, bgr)
        pruned, pts, cols, kps = ctx.pruner_prune(0.01, (case["H"], case["W"]))
        # the buffers that the call fills, whole: their first count rows are the points
        return {"pruned": pruned, "count": len(pts), "points": pts.base, "colors": cols.base, "keypts": kps.base}
    ctx.image_put_thumbnail(1, s["frame"], (case["H"], case["W"]))
    return ctx.image_get(1)


# ---- the same in 64 bits

def exact(case, seed):
    kind = case["kind"]
    if kind == "score":
        return _exact_score(case, seed)
    if kind == "clean":
        w = _window(case, seed)
        return _exact_clean(w["depths"], w["poses"], 0.01, MIN_CONSISTENT)
    if kind == "fuse":
        w = _window(case, seed)
        # the points are rows in raster order: one pixel decided otherwise, at a threshold, shifts all that follow
        pruned = _exact_prune(w["depths"], w["poses"], 0.01)
        return {"pruned": pruned, "count": None, "points": None, "colors": None, "keypts": None}
    # the others choose among planes by their scores, or are whole numbers
    return None


def _bearings64(W, H):
    return torch.from_numpy(synth.bearings(W, H))


def _exact_score(case, seed):
    p = _params(case, seed)
    seq, plane, _ = _score_inputs(case, seed)
    W, H, n, h = case["W"], case["H"], case["views"], p.patch_half
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    B = _bearings64(W, H).to(dev)
    P = torch.from_numpy(plane[..., :3].astype(np.float64)).to(dev)
    imgs = [torch.from_numpy(seq["images"][k]).to(dev).double() for k in range(n + 1)]
    ks = range(-h, h + 1, p.patch_stride)
    r0, r1, c0, c1 = h + 1, H - h, h + 1, W - h
    Pi = P[r0:r1, c0:c1]
    Ic = imgs[0][r0:r1, c0:c1]
    w, xs = [], []
    for k1 in ks:
        for k2 in ks:
            x = imgs[0][r0 + k1:r1 + k1, c0 + k2:c1 + k2]
            w.append(torch.exp(-(x - Ic) ** 2 / (2.0 * p.sigma_color ** 2) - (k1 * k1 + k2 * k2) / (2.0 * p.sigma_space ** 2)))
            xs.append(x)
    w, xs = torch.stack(w), torch.stack(xs)
    w = w / w.sum(0)
    mx = (w * xs).sum(0)
    vx = (w * (xs - mx) ** 2).sum(0)
    R0, t0 = seq["poses"][0][:9].reshape(3, 3), seq["poses"][0][9:]
    per_view = []
    for v in range(n):
        Rn, tn = seq["poses"][1 + v][:9].reshape(3, 3), seq["poses"][1 + v][9:]
        M = Rn @ R0.T
        c = torch.from_numpy(tn - M @ t0).to(dev)
        M = torch.from_numpy(M).to(dev)
        ys = []
        for k1 in ks:
            for k2 in ks:
                b = B[r0 + k1:r1 + k1, c0 + k2:c1 + k2]
                s = (b * Pi).sum(-1)
                s = torch.where(s < 0, -1.0, 1.0) * s.abs().clamp_min(1e-6)
                X = (b / s[..., None]) @ M.T + c
                u = torch.atan2(X[..., 0], X[..., 2]) * (W / (2 * math.pi)) + 0.5 * W
                y = torch.atan2(X[..., 1], torch.hypot(X[..., 0], X[..., 2])) * (H / math.pi) + 0.5 * H
                ys.append(_sample64(imgs[1 + v], u, y, p.edge_mode))
        ys = torch.stack(ys)
        my = (w * ys).sum(0)
        vy = (w * (ys - my) ** 2).sum(0)
        cov = (w * (xs - mx) * (ys - my)).sum(0)
        ncc = (cov / torch.sqrt((vx * vy).clamp_min(1e-30))).clamp(-1.0, 1.0)
        per_view.append(torch.where((vx < p.var_floor) | (vy < p.var_floor), torch.full_like(ncc, -1.0), ncc))
    k = max(1, min(p.topk, n))
    best = torch.stack(per_view).sort(0, descending=True).values[:k].mean(0)
    score = torch.zeros(H, W, dtype=torch.float64)
    score[r0:r1, c0:c1] = best.cpu()
    nrm = -P / P.norm(dim=-1, keepdim=True).clamp_min(1e-30)
    return {"score": score, "normals": nrm.cpu()}


def _sample64(img, u, v, edge):
    H, W = img.shape
    inside = torch.ones_like(u, dtype=torch.bool)
    if edge == pm.EDGE_ZERO:
        inside = (u >= 0) & (u < W - 1) & (v >= 0) & (v < H - 1)
    uu = u.clamp(0, W if edge == pm.EDGE_WRAP else W - 1)
    vv = v.clamp(0, H - 1)
    x, y = uu.floor(), vv.floor()
    fx, fy = uu - x, vv - y
    x, y = x.long(), y.long()
    x0, x1 = (x % W, (x + 1) % W) if edge == pm.EDGE_WRAP else (x, (x + 1).clamp(max=W - 1))
    y1 = (y + 1).clamp(max=H - 1)
    top = img[y, x0] * (1 - fx) + img[y, x1] * fx
    bot = img[y1, x0] * (1 - fx) + img[y1, x1] * fx
    return torch.where(inside, top * (1 - fy) + bot * fy, torch.zeros_like(u))


def _world64(B, pose, d):
    return (d[..., None] * B - pose[9:]) @ pose[:9].reshape(3, 3)


def _project64(X, pose, W, H):
    c = X @ pose[:9].reshape(3, 3).T + pose[9:]
    r = np.sqrt((c ** 2).sum(-1))
    near = r * r < 1e-8
    r = np.where(near, 1.0, r)
    y = H * (0.5 + np.arcsin(np.clip(c[..., 1] / r, -1, 1)) / np.pi)
    x = W * (0.5 + np.arctan2(c[..., 0], c[..., 2]) / (2 * np.pi))
    return x, y, r, near


def _exact_clean(depths, poses, thr, min_consistent):
    H, W = depths[0].shape
    d0 = depths[0].astype(np.float64)
    X = _world64(synth.bearings(W, H), poses[0], d0)
    seen = np.ones((H, W), int)
    for d, pose in zip(depths[1:], poses[1:]):
        x, y, r, near = _project64(X, pose, W, H)
        ok = ~near & (x >= 0) & (x < W) & (y >= 0) & (y < H)
        x, y = np.where(ok, x, 0.0), np.where(ok, y, 0.0)
        edge = (x >= W - 1) | (y >= H - 1)
        ix, iy = np.minimum(x.astype(int), W - 2), np.minimum(y.astype(int), H - 2)
        fx, fy = x - ix, y - iy
        dd = d.astype(np.float64)
        top = (1 - fx) * dd[iy, ix] + fx * dd[iy, ix + 1]
        bot = (1 - fx) * dd[iy + 1, ix] + fx * dd[iy + 1, ix + 1]
        v = np.where(edge, 0.0, (1 - fy) * top + fy * bot)
        seen += ok & (np.abs(v - r) < r * thr)
    return np.where((d0 >= 1e-6) & (seen >= min_consistent), d0, 0.0)


def _exact_prune(depths, poses, thr):
    """The head's pixels in raster order against each later map: a pixel behind a map's value within thr is
    dropped, one in front of it zeroes that value for the pixels after it."""
    H, W = depths[0].shape
    d0 = depths[0].astype(np.float64)
    zero = d0 == 0
    filt = zero.copy()
    filt[2:, :] |= zero[1:-1, :]
    filt[:, 2:] |= zero[:, 1:-1]
    filt[:-1, :] |= zero[1:, :]
    filt[:, :-1] |= zero[:, 1:]
    alive = ~filt
    X = _world64(synth.bearings(W, H), poses[0], d0)
    raster = np.arange(H * W).reshape(H, W)
    for d, pose in zip(depths[1:], poses[1:]):
        x, y, r, near = _project64(X, pose, W, H)
        ok = alive & ~near & (x >= 0) & (x < W) & (y >= 0) & (y < H) & (r >= 1e-5)
        q = np.where(ok, y, 0).astype(int) * W + np.where(ok, x, 0).astype(int)
        v = d.astype(np.float64).reshape(-1)[q]
        ok &= (v != 0) & ~(np.abs(v - r) > thr * r)
        first = np.full(H * W, H * W)
        front = ok & (d0 < v)
        np.minimum.at(first, q[front], raster[front])
        alive &= ~(ok & (raster < first[q]))
    return np.where(alive, d0, 0.0)
