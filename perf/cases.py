"""The work that programs built on this package have it do, as timed cases.

One case is one call pattern at one size:

    image     ORB.extract of one host image: a camera thread of a live system
    images    ORB.extract_batch_dev of resident images of uneven sizes with tracked
              points as seeds: a recorded sequence or several rigs processed offline
    rig       RigBatch.run (captured graph): live, one rig frame with the stereo pass
              and everything read back, or throughput, many frames left on the device
    match     Matcher.KnnMatch + FilterRatio + FilterThreshold of host descriptors:
              two frames, or a frame against the descriptors of a map
    window    window_search_dev: local map points projected into the rig's cameras
    pose      pose_optimization of one new frame against fixed map points, the
              problem built anew as for every tracked frame
    bow       place recognition: BowVocabulary.transform of a frame, then DBowMatch
              against a keyframe
    residual  reprojection forward and backward (torch.autograd)
    local_ba  a local bundle adjustment, built, optimized and read back
    schur     full linearization and Schur complement of a large problem whose
              edges stay on the device

listed() holds the sizes of this repository's configurations and tests (640 x 480 and
1280 x 720 images, 500 to 4000 features, 5000 map points, 20k points with 150k
observations, 200k points with 1.5M) and ordinary live ones; draw() spreads the same
patterns over their ranges.  Inputs come from the seed alone.
"""
import math
import random
from types import SimpleNamespace

import numpy as np
import torch

from mcvslam_amd import BALinearizer, Context, Matcher, ORB, RigBatch, synth
from mcvslam_amd.api import BowVocabulary, dbow_match, window_search_dev
from mcvslam_amd.autograd import reprojection
from mcvslam_amd.ba import local_ba_linearizer, pose_optimization

DEV = "cuda"
F64 = torch.float64
RIG_SIZES = ((1280, 720), (1280, 720), (640, 480))


# ---------------------------------------------------------------------------
# the cases

def listed():
    return [
        # one camera thread: the smallest extraction of a live system
        {"name": "image_640x480", "kind": "image", "w": 640, "h": 480, "nf": 2000},
        # six images of uneven sizes with points tracked from the frames before
        {"name": "images_6_uneven", "kind": "images", "n": 6, "w": 1241, "h": 733, "nf": 1500, "seeds": 150},
        # one live rig frame: features, pair matches and stereo depths, read by the tracker
        {"name": "rig_live", "kind": "rig", "frames": 1, "nf_lo": 2000, "nf_hi": 2000, "host": True},
        # 64 rig frames of uneven keypoint counts per step, tuned once, results left in HBM
        {"name": "rig_64", "kind": "rig", "frames": 64, "nf_lo": 500, "nf_hi": 4000, "host": False},
        # two frames' descriptors
        {"name": "match_frames", "kind": "match", "nq": 2000, "nt": 2000},
        # a frame's descriptors against those of a map
        {"name": "match_map", "kind": "match", "nq": 4000, "nt": 48000},
        # 5000 map points into three cameras of 2000 keypoints
        {"name": "window_3_cameras", "kind": "window", "cams": 3, "points": 5000, "kps": 2000},
        # the pose of one tracked frame, four rounds of 15 iterations
        {"name": "pose_frame", "kind": "pose", "points": 2000, "obs": 1500},
        # one frame against the vocabulary and one keyframe
        {"name": "bow_frame", "kind": "bow", "k": 10, "L": 5, "n": 2000},
        # residuals and their gradient, 10 keyframes
        {"name": "residual_150k", "kind": "residual", "kf": 10, "points": 20000, "obs": 150000},
        # a local map after a new keyframe: 10 keyframes, 20k points, 150k edges
        {"name": "local_ba_150k", "kind": "local_ba", "kf": 10, "points": 20000, "obs": 150000, "iters": 5},
        # 50 keyframes, 200k points, 1.5M edges: one linearization and Schur complement
        {"name": "schur_1500k", "kind": "schur", "kf": 50, "points": 200000, "obs": 1500000},
    ]


def draw(rng):
    def span(a, b):  # log-uniform whole number of [a, b]
        return max(a, min(b, int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))))

    kind = rng.choice(["image", "images", "rig", "match", "window", "pose", "bow", "residual", "local_ba", "schur"])
    c = {"kind": kind}
    if kind == "image":
        c["w"] = rng.randint(320, 1920)
        c["h"] = max(240, min(1080, int(c["w"] * rng.uniform(0.5, 0.8))))
        c["nf"] = span(500, 4000)
    elif kind == "images":
        c["w"] = rng.randint(400, 1400)
        c["h"] = max(300, int(c["w"] * rng.uniform(0.5, 0.8)))
        c.update(n=span(2, 24), nf=span(500, 4000), seeds=rng.choice([0, rng.randint(1, 400)]))
    elif kind == "rig":
        c["host"] = rng.random() < 0.5
        c["frames"] = span(1, 4) if c["host"] else span(2, 64)
        c["nf_lo"] = span(500, 2000)
        c["nf_hi"] = rng.randint(c["nf_lo"], min(4000, 4500 - c["nf_lo"]))
    elif kind == "match":
        c.update(nq=span(100, 4000), nt=span(100, 48000))
    elif kind == "window":
        c.update(cams=rng.randint(1, 3), points=span(500, 20000), kps=span(500, 4000))
    elif kind == "pose":
        c["points"] = span(300, 4000)
        c["obs"] = int(c["points"] * rng.uniform(0.4, 0.8))
    elif kind == "bow":
        c.update(k=rng.randint(6, 12), L=rng.randint(3, 5), n=span(300, 4000))
    elif kind in ("residual", "local_ba"):
        c.update(kf=rng.randint(3, 20), points=span(1000, 30000))
        c["obs"] = int(c["points"] * c["kf"] * rng.uniform(0.35, 0.6))
        if kind == "local_ba":
            c["iters"] = rng.randint(3, 6)
    else:
        c.update(kf=rng.randint(10, 50), points=span(10000, 200000))
        c["obs"] = int(c["points"] * c["kf"] * rng.uniform(0.1, 0.15))
    return c


# ---------------------------------------------------------------------------
# inputs

def _gen(seed):
    return torch.Generator(DEV).manual_seed(int(seed))


def _views(seed, sizes, parallax=0.0):
    """One scene rendered once per size, as uint8 images on the device: 400 Gaussian
    blobs, 60 rectangles in painter's order and N(0, 3) noise (synth.blob_image's
    recipe).  With parallax, view v > 0 sees every blob and rectangle shifted left
    by a disparity of its own in [2, 2 + parallax] px, as the right camera does."""
    r = np.random.Generator(np.random.PCG64(int(seed)))
    g = _gen(seed)
    bx, by, br = r.random(400), r.random(400), r.random(60)
    sig, amp = r.uniform(2, 20, 400), r.uniform(40, 200, 400) * np.where(r.random(400) < 0.5, -1, 1)
    bd = 2 + parallax * r.random(400)
    rx, ry, rw, rh, rv = r.random(60), r.random(60), r.uniform(8, 120, 60), r.uniform(8, 120, 60), r.uniform(0, 255, 60)
    rd = (2 + parallax * br).round()
    out = []
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
    s = dev(sig)[:, None]
    for v, (w, h) in enumerate(sizes):
        sh, rsh = (bd, rd) if v and parallax else (0 * bd, 0 * rd)
        gx = torch.exp(-((torch.arange(w, device=DEV)[None] - dev(bx * w - sh)[:, None]) / s) ** 2 / 2)
        gy = torch.exp(-((torch.arange(h, device=DEV)[None] - dev(by * h)[:, None]) / s) ** 2 / 2)
        im = (gy * dev(amp)[:, None]).t().contiguous() @ gx
        for i in range(60):
            xa, ya = rx[i] * w - rsh[i], ry[i] * h
            im[max(0, int(ya)):max(0, int(ya + rh[i])), max(0, int(xa)):max(0, int(xa + rw[i]))] = rv[i]
        im += 3 * torch.randn(im.shape, generator=g, device=DEV, dtype=F64)
        out.append(im.clamp_(0, 255).round_().to(torch.uint8).contiguous())
    return out


def _uneven(c):
    """The image sizes of an `images` case, from w x h down, odd ones among them."""
    return [(max(320, c["w"] - 97 * (i % 5)), max(240, c["h"] - 53 * (i % 4))) for i in range(c["n"])]


def _descriptors(g, n):
    return torch.randint(0, 256, (n, 32), generator=g, device=DEV, dtype=torch.uint8)


def _flipped(g, d, most):
    """d with 0 .. most bits of every row flipped."""
    p = torch.randint(0, most + 1, (len(d), 1), generator=g, device=DEV) / 256.0
    bits = (torch.rand((len(d), 256), generator=g, device=DEV) < p).view(len(d), 32, 8)
    return d ^ (bits * (2 ** torch.arange(8, device=DEV))).sum(-1).to(torch.uint8)


def _edges(seed, kf, points, obs, stereo=0.0, fixed=0.0, jitter=0.0, turn=0.0):
    """A multi-camera problem as synth.local_ba_problem describes it: keyframes along x,
    points in a box ahead of the rig, `obs` of the visible (point, keyframe, camera)
    triples with N(0, 1) px noise and 5 % outliers, the share `stereo` of the left
    camera's as stereo edges, the share `fixed` of the points fixed at their places,
    the other estimates moved by N(0, jitter) m and N(0, turn) rad and m."""
    g = _gen(seed)
    rand = lambda *s: torch.rand(s, generator=g, device=DEV, dtype=F64)
    randn = lambda *s: torch.randn(s, generator=g, device=DEV, dtype=F64)
    cams = synth.rig_cameras()
    f32 = lambda v: float(np.float32(v))
    table = np.array([[f32(c.fx), f32(c.fy), f32(c.cx), f32(c.cy), 0, 0, 0, 1, -c.baseline_x, 0, 0,
                       f32(math.sqrt(5.991))] for c in cams])
    yaw = (rand(kf) * 10 - 5) * math.pi / 180
    R, t = _rot_z(yaw), torch.zeros(kf, 3, device=DEV, dtype=F64)
    pos = torch.zeros(kf, 3, device=DEV, dtype=F64)
    pos[:, 0] = 0.3 * torch.arange(kf, device=DEV)
    t = -(R @ pos[:, :, None])[:, :, 0]
    X = rand(points, 3) * torch.tensor([10 + 0.3 * kf, 10.0, 5.0], device=DEV, dtype=F64)
    X += torch.tensor([-5.0, -5.0, 4.0], device=DEV, dtype=F64)
    seen, uvs, zs = [], [], []
    for f in range(kf):
        Pb = X @ R[f].t() + t[f]
        for k, c in enumerate(cams):
            x = Pb[:, 0] - c.baseline_x
            u, v = table[k, 0] * x / Pb[:, 2] + table[k, 2], table[k, 1] * Pb[:, 1] / Pb[:, 2] + table[k, 3]
            ok = ((Pb[:, 2] > 0.5) & (u >= 0) & (u < c.width) & (v >= 0) & (v < c.height)).nonzero()[:, 0]
            seen.append((ok * kf + f) * 3 + k)
            uvs.append(torch.stack([u, v], 1)[ok])
            zs.append(Pb[ok, 2])
    seen, uv, z = torch.cat(seen), torch.cat(uvs), torch.cat(zs)
    keep = torch.randperm(len(seen), generator=g, device=DEV)[:obs]
    seen, order = seen[keep].sort()
    uv, z = uv[keep][order], z[keep][order]
    cam, fr, pt = seen % 3, seen // 3 % kf, seen // (3 * kf)
    m = len(seen)
    size = torch.tensor([[c.width, c.height] for c in cams], device=DEV, dtype=F64)[cam]
    uv = uv + randn(m, 2)
    uv = torch.where(rand(m, 1) < 0.05, rand(m, 2) * size, uv)
    level = torch.randint(0, 8, (m,), generator=g, device=DEV)
    isig = torch.from_numpy((1 / np.float32(1.2) ** (2 * np.arange(8))).astype(np.float32)).to(DEV)[level]
    bf = f32(table[0, 0])
    ur = uv[:, 0] - bf / z + randn(m)
    ur = torch.where(rand(m) < 0.05, rand(m) * cams[0].width, ur)
    st = (cam == 0) & (rand(m) < stereo)
    hold = rand(points) < fixed
    Xe = X + torch.where(hold, 0.0, jitter)[:, None] * randn(points, 3)
    xi = turn * randn(kf, 6)
    if kf > 1:
        xi[0] = 0
    dR, dt = _exp(xi)
    Re, te = dR @ R, (dR @ t[:, :, None])[:, :, 0] + dt
    h = lambda a, d: np.ascontiguousarray(a.cpu().numpy(), d)
    frames = _frames(Re, te)
    mono = ~st
    ff = np.zeros(kf, np.int32)
    ff[0] = 1 if kf > 1 else 0
    Xh = h(Xe, np.float64)
    M = synth.BAProblem(h(uv[mono], np.float32), h(pt[mono], np.int32), h(fr[mono], np.int32), h(cam[mono], np.int32),
                        h(level[mono], np.int32), h(isig[mono], np.float32), Xh, frames, table, ff)
    S = None
    if stereo > 0:
        S = synth.StereoProblem(h(torch.cat([uv, ur[:, None]], 1)[st], np.float32), h(pt[st], np.int32),
                                h(fr[st], np.int32), h(isig[st], np.float32), Xh, frames,
                                np.array([*table[0, :4], bf, f32(math.sqrt(7.815))]))
    return M, S, h(hold, np.int32)


def _rot_z(a):
    R = torch.zeros(len(a), 3, 3, device=DEV, dtype=F64)
    R[:, 0, 0] = R[:, 1, 1] = torch.cos(a)
    R[:, 0, 1], R[:, 1, 0] = -torch.sin(a), torch.sin(a)
    R[:, 2, 2] = 1
    return R


def _skew(w):
    S = torch.zeros(len(w), 3, 3, device=w.device, dtype=F64)
    S[:, 0, 1], S[:, 0, 2], S[:, 1, 2] = -w[:, 2], w[:, 1], -w[:, 0]
    return S - S.transpose(1, 2)


def _exp(xi):
    """SE(3) exponentials (rotation first) of the rows of xi."""
    W = _skew(xi[:, :3])
    th = xi[:, :3].norm(dim=1).clamp_min(1e-12)[:, None, None]
    small, I = th < 1e-5, torch.eye(3, device=xi.device, dtype=F64)
    a = torch.where(small, 1.0, torch.sin(th) / th)
    b = torch.where(small, 0.5, (1 - torch.cos(th)) / th ** 2)
    c = torch.where(small, 1 / 6, (th - torch.sin(th)) / th ** 3)
    return I + a * W + b * W @ W, ((I + b * W + c * W @ W) @ xi[:, 3:, None])[:, :, 0]


def _frames(R, t):
    """(qx qy qz qw tx ty tz) of poses whose rotations are below 180 degrees, w >= 0."""
    w = 0.5 * torch.sqrt((1 + R[:, 0, 0] + R[:, 1, 1] + R[:, 2, 2]).clamp_min(1e-12))
    q = torch.stack([R[:, 2, 1] - R[:, 1, 2], R[:, 0, 2] - R[:, 2, 0], R[:, 1, 0] - R[:, 0, 1]], 1) / (4 * w[:, None])
    return torch.cat([q, w[:, None], t], 1).cpu().numpy()


def _vocabulary(seed, k, L):
    """A k-ary vocabulary of depth L, every child its parent with 24 bits flipped."""
    g = _gen(seed)
    rows, last = [torch.zeros(1, 32, device=DEV, dtype=torch.uint8)], None
    for l in range(1, L + 1):
        if l == 1:
            last = _descriptors(g, k)
        else:
            d = last.repeat_interleave(k, 0)
            pick = torch.rand((len(d), 256), generator=g, device=DEV).argsort(1) < 24
            last = d ^ (pick.view(-1, 32, 8) * (2 ** torch.arange(8, device=DEV))).sum(-1).to(torch.uint8)
        rows.append(last)
    n, leaves = sum(len(r) for r in rows), k ** L
    inner = n - leaves
    ptr = np.minimum(np.arange(n + 1) * k, n - 1).astype(np.int32)
    word = np.concatenate([-np.ones(inner, np.int32), np.arange(leaves, dtype=np.int32)])
    r = np.random.Generator(np.random.PCG64(int(seed)))
    weight = np.concatenate([np.zeros(inner), r.uniform(0.5, 4.0, leaves) * (r.random(leaves) >= 0.02)])
    desc = torch.cat(rows)
    return synth.Vocabulary(k, L, desc.cpu().numpy(), ptr, np.arange(1, n, dtype=np.int32), word, weight), last


def _context():
    """A context whose work is ordered with the program's torch work."""
    ctx = Context(0)
    ctx.use_torch_stream()
    return ctx


class _Held:
    """A buffer of a rig or linearizer as torch sees it: the tensor keeps its owner alive."""

    def __init__(self, owner, ptr, rows, width):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (rows, width), "typestr": "|u1", "data": (ptr, False),
                                         "strides": None, "version": 3}


def _held(owner, ptr, rows, width, dtype):
    return torch.as_tensor(_Held(owner, ptr, rows, width), device=DEV).view(dtype)


def prepare(case, seed):
    c, kind = SimpleNamespace(**case), case["kind"]
    s = SimpleNamespace(c=c, kind=kind)
    if kind == "image":
        s.orb = ORB(c.nf, ctx=_context())
        s.image = _views(seed, [(c.w, c.h)])[0].cpu().numpy()
        s.cap = s.orb.capacity(c.w, c.h)
    elif kind == "images":
        s.orb = ORB(c.nf, ctx=_context())
        s.images = [_views(seed + 7919 * i, [z])[0] for i, z in enumerate(_uneven(case))]
        s.seeds = None
        if c.seeds:
            r = np.random.Generator(np.random.PCG64(int(seed)))
            s.seeds = []
            for w, h in _uneven(case):  # at level coordinates, as the extractor appends them to their octave
                k = np.zeros(c.seeds, [("x", "<f4"), ("y", "<f4"), ("size", "<f4"), ("angle", "<f4"),
                                       ("response", "<f4"), ("octave", "<i4")])
                k["octave"] = r.integers(0, 4, c.seeds)
                sc = np.float32(1.2) ** k["octave"]
                k["x"] = 25 + r.random(c.seeds) * (w / sc - 50)
                k["y"] = 25 + r.random(c.seeds) * (h / sc - 50)
                k["size"], k["response"] = 31, r.integers(7, 200, c.seeds)
                s.seeds.append(k)
    elif kind == "rig":
        n = c.frames
        s.images = []
        for f in range(n):
            s.images += _views(seed + 7919 * f, RIG_SIZES[:2], parallax=60.0)
            s.images += _views(seed + 7919 * f + 1, RIG_SIZES[2:])
        r = np.random.Generator(np.random.PCG64(int(seed)))
        nf = None
        if c.nf_lo < c.nf_hi:
            nf = r.integers(c.nf_lo, c.nf_hi + 1, 3 * n)
            nf[r.integers(3 * n)] = c.nf_hi
        s.rig = RigBatch(ORB(c.nf_lo, ctx=_context()), n, nfeatures=nf)
        s.ptrs = [im.data_ptr() for im in s.images]
        if not c.host:
            s.rig.autotune(s.ptrs, reps=2)
            cap = s.rig.cap
            view = lambda p, w, dt: _held(s.rig, p, 3 * n * cap, w, dt).view(3 * n, cap, -1)
            count = lambda p: _held(s.rig, p, 3 * n, 4, torch.int32).view(-1)
            s.out = {"kps": view(s.rig.d_kps, 24, torch.float32), "desc": view(s.rig.d_desc, 32, torch.uint8),
                     "counts": count(s.rig.d_counts), "matches": view(s.rig.d_matches, 12, torch.int32),
                     "mcounts": count(s.rig.d_mcounts), "knn": view(s.rig.d_knn, 16, torch.int32)}
            for t in s.out.values():  # rows past an image's count stay as they are: zero
                t.zero_()
    elif kind == "match":
        g = _gen(seed)
        t = _descriptors(g, c.nt)
        q = _flipped(g, t[torch.randint(0, c.nt, (c.nq,), generator=g, device=DEV)], 40)
        new = torch.rand((c.nq, 1), generator=g, device=DEV) < 0.4
        s.ctx, s.q, s.t = _context(), torch.where(new, _descriptors(g, c.nq), q).cpu().numpy(), t.cpu().numpy()
    elif kind == "window":
        g = _gen(seed)
        s.ctx = _context()
        cams = synth.rig_cameras()[:c.cams]
        s.points = torch.rand((c.points, 3), generator=g, device=DEV) * torch.tensor([10.0, 10, 5], device=DEV)
        s.points -= torch.tensor([5.0, 5, -2], device=DEV)
        s.pdesc = _descriptors(g, c.points)
        s.plevel = torch.randint(0, 8, (c.points,), generator=g, device=DEV, dtype=torch.int32)
        s.Rt = np.array([[1, 0, 0, 0, 1, 0, 0, 0, 1, -k.baseline_x, 0, 0] for k in cams], np.float32)
        s.K = np.array([[k.fx, k.fy, k.cx, k.cy] for k in cams], np.float32)
        s.sizes = np.array([[k.width, k.height] for k in cams], np.int32)
        s.scales = (np.float32(1.2) ** np.arange(8)).astype(np.float32)
        s.kxy, s.kdesc = [], []
        for k in cams:  # 70 % noisy reprojections with 0 .. 30 bits flipped, the others anywhere
            x, y, z = s.points[:, 0] - k.baseline_x, s.points[:, 1], s.points[:, 2]
            uv = torch.stack([k.fx * x / z + k.cx, k.fy * y / z + k.cy], 1)
            size = torch.tensor([k.width, k.height], device=DEV)
            vis = ((uv >= 0) & (uv < size)).all(1).nonzero()[:, 0]
            pick = vis[torch.randperm(len(vis), generator=g, device=DEV)][:int(0.7 * c.kps)]
            near = uv[pick] + torch.randn((len(pick), 2), generator=g, device=DEV)
            rest = c.kps - len(pick)
            xy = torch.cat([near, torch.rand((rest, 2), generator=g, device=DEV) * size])
            d = torch.cat([_flipped(g, s.pdesc[pick], 30), _descriptors(g, rest)])
            order = torch.randperm(c.kps, generator=g, device=DEV)
            s.kxy.append(torch.minimum(xy.clamp_min(0), size - 1e-3)[order].contiguous())
            s.kdesc.append(d[order].contiguous())
    elif kind == "pose":
        s.ctx = _context()
        s.mono, s.stereo, _ = _edges(seed, 1, c.points, c.obs, stereo=0.5, turn=0.02)
        s.fixed = np.ones(c.points, np.int32)
    elif kind == "bow":
        voc, leaves = _vocabulary(seed, c.k, c.L)
        s.voc = BowVocabulary(voc, _context())
        g = _gen(seed + 1)
        take = lambda: leaves[torch.randint(0, len(leaves), (c.n,), generator=g, device=DEV)]
        base = take()
        s.desc = _flipped(g, base, 30).cpu().numpy()
        old = torch.where(torch.rand((c.n, 1), generator=g, device=DEV) < 0.5, base, take())
        s.key_desc = _flipped(g, old, 30).cpu().numpy()
        s.key_fv = s.voc.transform(s.key_desc)[2]
    elif kind == "residual":
        s.mono, _, _ = _edges(seed, c.kf, c.points, c.obs)
        s.lin = BALinearizer.from_problem(s.mono, ctx=_context())
        g = _gen(seed + 1)
        s.dpose = (1e-3 * torch.randn((c.kf, 6), generator=g, device=DEV)).requires_grad_()
        s.dpoint = (1e-3 * torch.randn((c.points, 3), generator=g, device=DEV)).requires_grad_()
        s.grad = torch.randn((len(s.mono.obs_pt), 2), generator=g, device=DEV)
    elif kind == "local_ba":
        s.ctx = _context()
        s.mono, s.stereo, s.fixed = _edges(seed, c.kf, c.points, c.obs, 0.3, 0.1, 0.05, 0.01)
    else:
        s.mono, _, _ = _edges(seed, c.kf, c.points, c.obs)
        s.lin = BALinearizer.from_problem(s.mono, ctx=_context())
        ptr, m = s.lin.planes_ptr()
        s.planes = _held(s.lin, ptr, 22, 4 * m, torch.float32)
    return s


# ---------------------------------------------------------------------------
# one pass

def _filled(a, n):
    """The rows of a in an array of n rows, as a program keeps them in its frames' own buffers."""
    out = np.zeros((n,) + a.shape[1:], a.dtype)
    out[:len(a)] = a
    return out


def _fields(k):
    return {"xysar": np.stack([k[f] for f in ("x", "y", "size", "angle", "response")], -1), "octave": k["octave"]}


def run(s):
    c, kind = s.c, s.kind
    if kind == "image":
        kps, desc = s.orb.extract(s.image)
        return {"kps": _fields(_filled(kps, s.cap)), "desc": _filled(desc, s.cap), "count": len(kps)}
    if kind == "images":
        kps, desc, counts = s.orb.extract_batch_dev(s.images, seeds=s.seeds)
        return {"kps": kps, "desc": desc, "counts": counts}
    if kind == "rig":
        s.rig.run(s.ptrs)
        if not c.host:
            return s.out
        stereo = s.rig.stereo(2388.0, 1.0)
        kps, desc, counts, matches, mcounts, knn = s.rig.read()
        pairs = counts.reshape(-1, 3)[:, [0, 2, 2]].reshape(-1)  # the pairs' query images: L, W, W
        for rows, n in [(kps, counts), (desc, counts), (knn, pairs), (matches, mcounts)] + [(a, counts[::3]) for a in stereo]:
            for a, k in zip(rows, n):
                a[k:] = 0  # nothing is written there
        return {"kps": _fields(kps), "desc": desc, "counts": counts, "knn": knn, "matches": matches,
                "mcounts": mcounts, "u_right": stereo[0], "depth": stereo[1], "sad": stereo[2]}
    if kind == "match":
        knn = Matcher.KnnMatch(s.q, s.t, ctx=s.ctx)
        m = knn.FilterRatio(0.7).FilterThreshold(50)
        return {"knn": knn.rows, "matches": _filled(m, c.nq), "count": len(m)}
    if kind == "window":
        return window_search_dev(s.points, s.pdesc, s.plevel, s.Rt, s.K, s.sizes, s.scales, 15.0, 0.7, 50, s.kxy,
                                 s.kdesc, ctx=s.ctx)
    if kind == "pose":
        lin = local_ba_linearizer(s.mono, s.stereo, s.fixed, ctx=s.ctx)
        p = pose_optimization(lin)
        lin.close()
        # the frame keeps its pose as float (cv::Mat CV_32F)
        return {"frame": p.frames.astype(np.float32), "inliers": p.inliers,
                "active": np.concatenate([p.active_mono, p.active_stereo])}
    if kind == "bow":
        word, vec, fv = s.voc.transform(s.desc)
        m = dbow_match(s.desc, fv, s.key_desc, s.key_fv, ctx=s.voc.ctx)
        return {"word": word[0], "weight": word[1], "node": word[2], "vec_word": _filled(vec[0], c.n),
                "vec": _filled(vec[1], c.n), "fv": [_filled(a, c.n + 1) for a in fv], "matches": _filled(m, c.n)}
    if kind == "residual":
        e = reprojection(s.dpose, s.dpoint, s.lin, (s.mono.points, s.mono.frames, s.mono.cams))
        gp, gx = torch.autograd.grad(e, (s.dpose, s.dpoint), s.grad)
        return {"e": e.detach(), "pose": gp, "point": gx}
    if kind == "local_ba":
        lin = local_ba_linearizer(s.mono, s.stereo, s.fixed, ctx=s.ctx)
        stats, _ = lin.optimize(c.iters)
        points, frames = lin.get_state()
        lin.close()
        # the map keeps positions and poses as float (cv::Mat CV_32F)
        return {"points": points.astype(np.float32), "frames": frames.astype(np.float32),
                "chi2": stats[:, :2].astype(np.float32)}
    s.lin.linearize()
    S, b = s.lin.schur(1e4)
    # the reduced system is computed in float and read as double
    return {"planes": s.planes, "S": S.astype(np.float32), "b": b.astype(np.float32)}


def work(case):
    c = SimpleNamespace(**case)
    kind, flops = c.kind, 0.0
    if kind == "image":
        return {"bytes": c.w * c.h + 56 * c.nf, "flops": 0}
    if kind == "images":
        return {"bytes": sum(w * h for w, h in _uneven(case)) + 56 * c.n * (c.nf + c.seeds), "flops": 0}
    if kind == "rig":
        nf = (c.nf_lo + c.nf_hi) / 2
        rows = 56 + 16 + 6 + (4 if c.host else 0)  # keypoint, descriptor, knn row, about half a match, depths
        return {"bytes": c.frames * (sum(w * h for w, h in RIG_SIZES) + 3 * nf * rows),
                "flops": c.frames * 3 * nf * nf * 512}
    if kind == "match":  # a distance as a 256-term product
        return {"bytes": 32 * (c.nq + c.nt) + 22 * c.nq, "flops": 512.0 * c.nq * c.nt}
    if kind == "window":
        return {"bytes": 48 * c.points + c.cams * (40 * c.kps + 24 * c.points), "flops": c.cams * c.points * 40}
    if kind == "pose":  # the edges once per round (linearized at least once, then tested)
        return {"bytes": 24 * c.points + 4 * 25 * c.obs, "flops": 4 * 400.0 * c.obs}
    if kind == "bow":
        return {"bytes": c.n * (64 + 16 + 20 + 8) + 32 * min(c.n * c.k * c.L, c.k ** c.L), "flops": c.n * c.k * c.L * 512}
    if kind == "residual":
        return {"bytes": c.obs * (20 + 8 + 8) + c.points * (24 + 24), "flops": 500.0 * c.obs}
    if kind == "local_ba":  # per iteration: the edges twice (linearized, then the trial's residuals), the points twice
        return {"bytes": c.iters * (2 * 20 * c.obs + 48 * c.points), "flops": c.iters * 1500.0 * c.obs}
    return {"bytes": c.obs * (20 + 88) + c.points * 24 + (6 * c.kf) ** 2 * 8, "flops": 1500.0 * c.obs}


# ---------------------------------------------------------------------------
# the same values in 64 bits

class _Problem:
    """The edges of _edges() as 64-bit tensors, linearized and reduced in plain torch."""

    def __init__(self, M, S=None, hold=None):
        d = lambda a, dt=F64: torch.as_tensor(np.asarray(a)).to(DEV, dt)
        self.uv, self.isig = d(M.obs_uv), d(M.obs_isig)
        self.pt, self.fr, self.cam = (d(a, torch.int64) for a in (M.obs_pt, M.obs_frame, M.obs_cam))
        self.K = d(M.cams)[:, :4]
        self.tc, self.delta = d(M.cams)[:, 8:11], d(M.cams)[:, 11]
        self.X, self.frames0 = d(M.points), np.asarray(M.frames)
        q = d(M.frames)[:, :4]
        v = q[:, :3]
        W = _skew(v)
        self.R = torch.eye(3, device=DEV, dtype=F64) + 2 * q[:, 3, None, None] * W + 2 * W @ W
        self.t = d(M.frames)[:, 4:]
        self.hold = d(hold if hold is not None else np.zeros(len(self.X)), torch.bool)
        self.free = (d(M.frame_fixed, torch.int64) == 0).nonzero()[:, 0]
        self.S = None
        if S is not None:
            self.S = SimpleNamespace(obs=d(S.obs), pt=d(S.obs_pt, torch.int64), fr=d(S.obs_frame, torch.int64),
                                     isig=d(S.obs_isig), cam=[float(np.float32(x)) for x in S.cam])
        n = [len(self.pt)] + ([len(self.S.pt)] if S is not None else [])
        self.active = [torch.ones(k, device=DEV, dtype=torch.bool) for k in n]
        self.robust = True

    def _weigh(self, chi2, delta):
        w = torch.where(chi2 <= delta ** 2, 1.0, delta / chi2.clamp_min(1e-300).sqrt())
        rho = torch.where(chi2 <= delta ** 2, chi2, 2 * chi2.sqrt() * delta - delta ** 2)
        return (w, rho) if self.robust else (torch.ones_like(w), chi2)

    def mono(self):
        """e, chi2, w, rho, J_pose, J_point of the mono edges."""
        R, K, P = self.R[self.fr], self.K[self.cam], self.X[self.pt]
        Pb = (R @ P[:, :, None])[:, :, 0] + self.t[self.fr]
        x, y, z = (Pb + self.tc[self.cam]).unbind(1)
        e = self.uv - torch.stack([K[:, 0] * x / z + K[:, 2], K[:, 1] * y / z + K[:, 3]], 1)
        chi2 = self.isig * (e ** 2).sum(1)
        J = torch.zeros(len(x), 2, 3, device=DEV, dtype=F64)
        J[:, 0, 0], J[:, 0, 2] = K[:, 0] / z, -K[:, 0] * x / z ** 2
        J[:, 1, 1], J[:, 1, 2] = K[:, 1] / z, -K[:, 1] * y / z ** 2
        w, rho = self._weigh(chi2, self.delta[self.cam])
        return e, chi2, w, rho, torch.cat([J @ _skew(Pb), -J], 2), -J @ R

    def stereo(self):
        s, (fx, fy, cx, cy, bf, delta) = self.S, self.S.cam
        R = self.R[s.fr]
        C = (R @ self.X[s.pt][:, :, None])[:, :, 0] + self.t[s.fr]
        x, y, z = C.unbind(1)
        i32 = (1 / z).float()  # the edge rounds the inverse depth and its product with bf to float
        iz = i32.to(F64)
        u = x * iz * fx + cx
        e = s.obs - torch.stack([u, y * iz * fy + cy, u - (np.float32(bf) * i32).to(F64)], 1)
        chi2 = s.isig * (e ** 2).sum(1)
        J = torch.zeros(len(x), 3, 3, device=DEV, dtype=F64)
        J[:, 0, 0] = J[:, 2, 0] = fx / z
        J[:, 1, 1], J[:, 1, 2] = fy / z, -fy * y / z ** 2
        J[:, 0, 2] = -fx * x / z ** 2
        J[:, 2, 2] = J[:, 0, 2] + bf / z ** 2
        w, rho = self._weigh(chi2, torch.tensor(delta, device=DEV, dtype=F64))
        return e, chi2, w, rho, torch.cat([J @ _skew(C), -J], 2), -J @ R

    def edges(self):
        out = [(self.mono(), self.pt, self.fr, self.isig, self.active[0])]
        if self.S is not None:
            out.append((self.stereo(), self.S.pt, self.S.fr, self.S.isig, self.active[1]))
        return out

    def chi2(self):
        return float(sum(v[3][a].sum() for v, _, _, _, a in self.edges()))

    def blocks(self):
        """H_pp, b_p per frame, H_ll, b_l per point, and H_pl as [points][frames][6][3] (a generator over chunks)."""
        F, P = len(self.R), len(self.X)
        z = lambda *n: torch.zeros(*n, device=DEV, dtype=F64)
        Hp, bp, Hl, bl = z(F, 6, 6), z(F, 6), z(P, 3, 3), z(P, 3)
        parts = []
        for (e, _, w, _, Jp, Jx), pt, fr, isig, act in self.edges():
            W = (w * isig * act)[:, None, None]
            live = ~self.hold[pt]
            Hp.index_add_(0, fr, Jp.transpose(1, 2) @ (W * Jp))
            bp.index_add_(0, fr, -(Jp.transpose(1, 2) @ (W * e[:, :, None]))[:, :, 0])
            Wl = W * live[:, None, None]
            Hl.index_add_(0, pt, Jx.transpose(1, 2) @ (Wl * Jx))
            bl.index_add_(0, pt, -(Jx.transpose(1, 2) @ (Wl * e[:, :, None]))[:, :, 0])
            parts.append((pt, fr, Jp.transpose(1, 2) @ (Wl * Jx)))
        seen = z(P).bool()
        for (_, pt, _, _, act) in self.edges():
            seen[pt[act]] = True
        return Hp, bp, Hl, bl, parts, seen & ~self.hold

    def reduced(self, lam, B=None):
        """S, b_schur and the back-substitution's D^-1, b_l and H_pl chunks."""
        Hp, bp, Hl, bl, parts, used = B or self.blocks()
        F, P, fi, n = len(self.R), len(self.X), self.free, 6 * len(self.free)
        I3 = torch.eye(3, device=DEV, dtype=F64)
        Di = torch.linalg.inv(torch.where(used[:, None, None], Hl + lam * I3, I3)) * used[:, None, None]
        S = torch.zeros(n, n, device=DEV, dtype=F64)
        for k, f in enumerate(fi.tolist()):
            S[6 * k:6 * k + 6, 6 * k:6 * k + 6] = Hp[f] + lam * torch.eye(6, device=DEV, dtype=F64)
        b = bp[fi].reshape(-1).clone()
        chunks = []
        step = max(1, 40_000_000 // max(1, F * 18))
        for p0 in range(0, P if n else 0, step):
            p1 = min(P, p0 + step)
            H = torch.zeros((p1 - p0) * F, 6, 3, device=DEV, dtype=F64)
            for pt, fr, h in parts:
                m = (pt >= p0) & (pt < p1)
                H.index_add_(0, (pt[m] - p0) * F + fr[m], h[m])
            A = H.view(p1 - p0, F, 6, 3)[:, fi].permute(1, 2, 0, 3).reshape(n, p1 - p0, 3)
            Y = (A.permute(1, 0, 2) @ Di[p0:p1]).permute(1, 0, 2).reshape(n, -1)
            S -= Y @ A.reshape(n, -1).t()
            b -= Y @ bl[p0:p1].reshape(-1)
            chunks.append((p0, p1, A))
        return S, b, Di, bl, chunks, Hp, bp, Hl, used

    def optimize(self, iterations, tau=1e-5, max_trials=10):
        """g2o's Levenberg-Marquardt; rows (chi2 before, chi2 after) per iteration."""
        stats, lam, ni = [], 0.0, 2.0
        fi = self.free
        for it in range(iterations):
            chi = self.chi2()
            row = [chi, chi]
            B = self.blocks()
            if it == 0:
                d = [B[0][fi].diagonal(dim1=1, dim2=2).reshape(-1), B[2][B[5]].diagonal(dim1=1, dim2=2).reshape(-1)]
                lam = tau * float(torch.cat(d).abs().max())
            trials, rho = 0, 0.0
            while True:
                keep = self.R, self.t, self.X
                S, b, Di, bl, chunks, *_ = self.reduced(lam, B)
                x = torch.linalg.solve(S, b) if len(b) else b
                c = bl.clone()
                for p0, p1, A in chunks:
                    c[p0:p1] -= (x @ A.reshape(len(x), -1)).reshape(-1, 3)
                xl = (Di @ c[:, :, None])[:, :, 0]
                scale = float((x * (lam * x + B[1][fi].reshape(-1))).sum() + (xl * (lam * xl + bl)).sum()) + 1e-3
                dR, dt = _exp(x.reshape(-1, 6))
                self.R, self.t, self.X = self.R.clone(), self.t.clone(), self.X + xl
                self.R[fi], self.t[fi] = dR @ keep[0][fi], (dR @ keep[1][fi][:, :, None])[:, :, 0] + dt
                new = self.chi2()
                rho = (chi - new) / scale
                trials += 1
                if rho > 0 and math.isfinite(new):
                    lam *= max(1 / 3, min(2 / 3, 1 - (2 * rho - 1) ** 3))
                    ni, chi = 2.0, new
                    break
                self.R, self.t, self.X = keep
                lam *= ni
                ni *= 2
                if not rho < 0 or trials >= max_trials or not math.isfinite(lam):
                    break
            row[1] = chi
            stats.append(row)
            if trials == max_trials or rho == 0 or not math.isfinite(lam):
                break
        return np.array(stats)

    def frames(self):
        return _frames(self.R, self.t)


def exact(case, seed):
    c, kind = SimpleNamespace(**case), case["kind"]
    if kind == "pose":
        M, S, _ = _edges(seed, 1, c.points, c.obs, stereo=0.5, turn=0.02)
        p = _Problem(M, S, np.ones(c.points))
        for r in range(4):
            p.optimize(15)
            bad = 0
            for k, (v, _, _, _, act) in enumerate(p.edges()):
                out = act & (v[1] >= 5.991)
                p.active[k] = act & ~out
                bad += int(out.sum())
            p.robust = p.robust and r != 2
            if len(M.obs_pt) + len(S.obs_pt) - bad < 10:
                break
        return {"frame": p.frames(), "inliers": None, "active": None}
    if kind == "bow":
        s = prepare(case, seed)
        voc, leaves = _vocabulary(seed, c.k, c.L)
        desc = torch.from_numpy(voc.desc).to(DEV)
        pop = torch.tensor([bin(i).count("1") for i in range(256)], device=DEV, dtype=torch.int16)
        d, node = torch.from_numpy(s.desc).to(DEV), torch.zeros(c.n, device=DEV, dtype=torch.int64)
        for _ in range(c.L):
            kids = node[:, None] * c.k + 1 + torch.arange(c.k, device=DEV)[None]
            dist = pop[(d[:, None] ^ desc[kids]).long()].sum(-1)
            best = (dist.long() * 64 + torch.arange(c.k, device=DEV)).argmin(1)
            node = kids[torch.arange(c.n, device=DEV), best]
        node = node.cpu().numpy()
        w = voc.weight[node]
        words = voc.word_id[node][w > 0]
        vec = np.bincount(words, w[w > 0], minlength=len(leaves))
        vec = vec[np.bincount(words, minlength=len(leaves)) > 0]
        return {"word": None, "weight": w, "node": None, "vec_word": None,
                "vec": _filled(vec / np.abs(vec).sum(), c.n), "fv": [None, None, None], "matches": None}
    if kind == "residual":
        s = prepare(case, seed)
        p = _Problem(s.mono)
        dR, dt = _exp(s.dpose.detach().double())
        p.R, p.t = dR @ p.R, (dR @ p.t[:, :, None])[:, :, 0] + dt
        p.X = p.X + s.dpoint.detach().double()
        e, _, _, _, Jp, Jx = p.mono()
        g = s.grad.double()[:, :, None]
        gp = torch.zeros(c.kf, 6, device=DEV, dtype=F64).index_add_(0, p.fr, (Jp.transpose(1, 2) @ g)[:, :, 0])
        gx = torch.zeros(c.points, 3, device=DEV, dtype=F64).index_add_(0, p.pt, (Jx.transpose(1, 2) @ g)[:, :, 0])
        return {"e": e, "pose": gp, "point": gx}
    if kind == "local_ba":
        M, S, hold = _edges(seed, c.kf, c.points, c.obs, 0.3, 0.1, 0.05, 0.01)
        p = _Problem(M, S, hold)
        stats = p.optimize(c.iters)
        return {"points": p.X, "frames": p.frames(), "chi2": stats}
    if kind == "schur":
        p = _Problem(_edges(seed, c.kf, c.points, c.obs)[0])
        e, chi2, w, _, Jp, Jx = p.mono()
        planes = torch.cat([e, chi2[:, None], w[:, None], Jp.reshape(-1, 12), Jx.reshape(-1, 6)], 1).t().contiguous()
        S, b = p.reduced(1e4)[:2]
        return {"planes": planes, "S": S, "b": b}
    return None
