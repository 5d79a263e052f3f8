"""The work that users of this framework have it do, as measurable cases.

Every case goes through the public entry points (the Python classes of
recon_amd, or the C ABI of include/rt_*.h where a program on the device calls
it), on synthetic RGB-D frames that are rendered on the GPU from a seed:
textured scenes at 0.3-7 m, 1 % sensor noise, motions as between a camera's
frames and its keyframe.

Kinds of cases:
  disparity   one Kinect disparity frame to depth (the sensor's input stage)
  pair        one keyframe and one frame on the single-pair tracker: keyframe
              preparation, frame preparation, coarse-to-fine tracking
  sequence    a frame sequence on the device with keyframe fusion
  pipeline    the sequence engine with learned warm starts
  batch       independent frame pairs in one call, all modes, one or mixed sizes
  learned     a batch whose pairs start from the pose network's proposals
  forward     the pose network's outputs (inference)
  gradient    the pose network's loss and gradients (training)
  tsdf        one frame fused into the voxel grid, and the grid's ray cast
"""
import ctypes
import math

import numpy as np
import torch

from recon_amd import BIOBJECTIVE, GEOMETRIC, PHOTOMETRIC, RtPair, check, lib, synth, synth_lib
from recon_amd.cnn import PoseNet, init_params, pose_to_target
from recon_amd.pipeline import SequenceTracker
from recon_amd.sensor import depth_mm_to_u16, disparity_to_depth
from recon_amd.tracker import BatchTracker, PhotoTracker
from recon_amd.tsdf import VoxelGrid, default_params

MODES = {"photometric": PHOTOMETRIC, "geometric": GEOMETRIC, "bi-objective": BIOBJECTIVE}
ITERS = (1, 3, 10, 5)          # coarse to fine, the reference's schedule
MIXED = ((160, 120), (320, 240), (480, 360), (640, 480))
# multiply-adds of the pose network's six convolutions per pair (4-32-64-128-128-256-256 at 80x60)
NET_MACS = 9 * (40 * 30 * 32 * 4 + 20 * 15 * 64 * 32 + 10 * 8 * 128 * 64 + 5 * 4 * 128 * 128 + 3 * 2 * 256 * 128 + 2 * 256 * 256)
NET_PARAMS = 1127910


def listed():
    return [
        # a capture loop converts every raw disparity frame before anything else sees it
        {"name": "disparity_640x480", "kind": "disparity", "width": 640, "height": 480, "half": True},
        # one keyframe switch and one tracked frame of a small live camera: latency
        {"name": "pair_320x240_photo", "kind": "pair", "width": 320, "height": 240, "mode": "photometric", "points": 8192},
        # the tracker's default mode (point-to-plane ICP), at VGA
        {"name": "pair_640x480_geo", "kind": "pair", "width": 640, "height": 480, "mode": "geometric", "points": 8192},
        # dense bi-objective tracking of a recorded VGA sequence with fused keyframes
        {"name": "sequence_640x480_bi", "kind": "sequence", "width": 640, "height": 480, "mode": "bi-objective",
         "points": 61440, "frames": 32, "interval": 10, "fuse": 5},
        # the whole engine on a live-like sequence: the network's warm start, tracking, fusion, keyframe policy
        {"name": "pipeline_640x480", "kind": "pipeline", "width": 640, "height": 480, "points": 61440, "frames": 24},
        # one frame against 64 keyframes, the batch that a relocalisation tracks
        {"name": "learned_64_640x480", "kind": "learned", "pairs": 64, "width": 640, "height": 480, "points": 8192},
        # a serving queue of cameras of different sizes
        {"name": "batch_256_mixed", "kind": "batch", "pairs": 256, "width": 0, "height": 0, "mode": "photometric",
         "points": 8192},
        # registration of frame pairs with both error terms
        {"name": "batch_64_320x240_bi", "kind": "batch", "pairs": 64, "width": 320, "height": 240,
         "mode": "bi-objective", "points": 8192},
        # the headline: large motions, proposals and tracking of a full batch
        {"name": "learned_4096_640x480", "kind": "learned", "pairs": 4096, "width": 640, "height": 480, "points": 8192},
        # inference over a full batch of prepared network inputs
        {"name": "forward_4096", "kind": "forward", "pairs": 4096},
        # one training batch
        {"name": "gradient_256", "kind": "gradient", "pairs": 256},
        # the voxel model's per-frame work at the reference's grid
        {"name": "tsdf_256_320x240", "kind": "tsdf", "resolution": 256, "width": 320, "height": 240},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def _size(rng, wmax=640, hmax=480):
    """An image size the trackers take: width a multiple of 16, height of 8."""
    return 16 * rng.randint(8, wmax // 16), 8 * rng.randint(12, hmax // 8)


def _points(rng, width, height, most):
    return 256 * _log_int(rng, 4, min(most, width * height // 2) // 256)


def draw(rng):
    kind = rng.choice(("disparity", "pair", "pair", "sequence", "pipeline", "batch", "batch", "learned", "forward",
                       "gradient", "tsdf", "tsdf"))
    if kind == "disparity":
        return {"kind": kind, "width": rng.randint(160, 1280), "height": rng.randint(120, 1024),
                "half": rng.random() < 0.5}
    if kind == "pair":
        w, h = _size(rng)
        return {"kind": kind, "width": w, "height": h, "mode": rng.choice(sorted(MODES)),
                "points": _points(rng, w, h, 61440)}
    if kind == "sequence":
        w, h = _size(rng)
        interval = rng.randint(4, 12)
        return {"kind": kind, "width": w, "height": h, "mode": rng.choice(sorted(MODES)),
                "points": _points(rng, w, h, 61440), "frames": rng.randint(8, 32), "interval": interval,
                "fuse": rng.randint(0, min(5, interval - 1))}
    if kind == "pipeline":
        w, h = rng.choice(((320, 240), (480, 360), (640, 480)))
        return {"kind": kind, "width": w, "height": h, "points": _points(rng, w, h, 61440), "frames": rng.randint(8, 24)}
    if kind == "batch":
        mixed = rng.random() < 0.4
        w, h = (0, 0) if mixed else (16 * rng.randint(10, 40), 8 * rng.randint(15, 60))
        mode = rng.choice(("photometric", "photometric", "bi-objective", "geometric"))
        return {"kind": kind, "pairs": _log_int(rng, 1, 256 if mode == "photometric" else 128), "width": w, "height": h,
                "mode": mode, "points": 8192}
    if kind == "learned":
        w, h = rng.choice(((160, 120), (320, 240), (640, 480)))
        return {"kind": kind, "pairs": _log_int(rng, 1, 2048), "width": w, "height": h, "points": 8192}
    if kind == "forward":
        return {"kind": kind, "pairs": _log_int(rng, 1, 4096)}
    if kind == "gradient":
        return {"kind": kind, "pairs": _log_int(rng, 8, 512)}
    return {"kind": kind, "resolution": 8 * rng.randint(8, 48), "width": rng.randint(96, 640),
            "height": rng.randint(80, 480)}


# ------------------------------------------------------------------ frames
def _render(scene, pose, width, height, seed, gray, depth, noise=0.01):
    fx, fy, cx, cy = synth.pinhole(width, height)
    T = np.ascontiguousarray(pose, np.float64).ravel()
    check(synth_lib().rs_render_device(scene, T.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), width, height, fx, fy,
                                       cx, cy, ctypes.c_uint64(seed), noise, gray, depth, None), "rs_render_device")


class _Scenes:
    def __init__(self, seed, count):
        self.h = [synth_lib().rs_scene_create(ctypes.c_uint64(seed * 1009 + k)) for k in range(count)]

    def free(self):
        torch.cuda.synchronize()
        for h in self.h:
            synth_lib().rs_scene_destroy(h)


def _frame_pairs(seed, sizes, theta, tmax):
    """Frame pairs of the given sizes in two device tensors (8-bit gray and
    16-bit depth, the keyframe before the frame): per pair the device pointers
    and calibration that the trackers take, and the true motion."""
    npx = [w * h for w, h in sizes]
    off = np.concatenate([[0], np.cumsum([2 * p for p in npx])])
    gray = torch.empty(int(off[-1]), dtype=torch.uint8, device="cuda")
    depth = torch.empty(int(off[-1]), dtype=torch.int16, device="cuda")
    scenes = _Scenes(seed, min(len(sizes), 64))
    cal = {s: synth.calib_block_np(*s) for s in set(sizes)}
    pairs, motions = [], []
    for i, (w, h) in enumerate(sizes):
        M = synth.sample_motion(seed * 100003 + i, theta, tmax)
        p = []
        for f, T in ((0, np.eye(4)), (1, M)):
            o = int(off[i]) + f * npx[i]
            g, d = gray.data_ptr() + o, depth.data_ptr() + 2 * o
            _render(scenes.h[i % len(scenes.h)], T, w, h, seed * 7919 + 2 * i + f, g, d)
            p += [g, d]
        pairs.append(dict(ref_gray=p[0], ref_depth=p[1], cur_gray=p[2], cur_depth=p[3], width=w, height=h,
                          calib=cal[(w, h)]))
        motions.append(M)
    scenes.free()
    return pairs, np.array(motions), (gray, depth)


def _sequence(seed, n, width, height, rot, trans, noise=0.01):
    poses = synth.trajectory(seed * 13 + 5, n, rot, trans, 0, 1.0)
    gray = torch.empty((n, height, width), dtype=torch.uint8, device="cuda")
    depth = torch.empty((n, height, width), dtype=torch.int16, device="cuda")
    scenes = _Scenes(seed, 1)
    for k in range(n):
        _render(scenes.h[0], poses[k], width, height, seed * 1000 + k, gray[k].data_ptr(), depth[k].data_ptr(), noise)
    scenes.free()
    return gray, depth, poses


class _Frames:
    """A device tensor as the buffer that SequenceTracker.run takes."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


class _Voxels:
    """A grid's voxels on the device, for torch.as_tensor (no copy)."""

    def __init__(self, grid):
        self.grid, r = grid, grid.res
        self.__cuda_array_interface__ = {"shape": (r, r, r, 2), "typestr": "<f4", "version": 2,
                                         "data": (lib().rt_tsdf_data(grid.h), False)}


def _net_inputs(seed, n, net):
    """The network's inputs of n rendered frame pairs, and the true motions."""
    pairs, motions, frames = _frame_pairs(seed, [(160, 120)] * n, 10.0, 150.0)
    x = torch.empty((n, net.cfg.in_height, net.cfg.in_width, net.cfg.channels[0]), dtype=torch.bfloat16, device="cuda")
    arr = (RtPair * n)()
    for i, p in enumerate(pairs):
        for k in ("ref_gray", "ref_depth", "cur_gray", "cur_depth", "width", "height"):
            setattr(arr[i], k, p[k])
    net.make_inputs(arr, n, x.data_ptr())
    torch.cuda.synchronize()
    return x, motions, frames


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    seed = int(seed) % (1 << 30)
    torch.cuda.init()
    if kind == "disparity":
        w, h = case["width"], case["height"]
        gen = torch.Generator(device="cuda").manual_seed(seed)
        # an uneven surface seen from the sensor: 11-bit disparities, with holes (2047)
        yy = torch.linspace(0, 6, h, device="cuda")[:, None] + torch.rand(1, device="cuda", generator=gen) * 6
        xx = torch.linspace(0, 8, w, device="cuda")[None, :] + torch.rand(1, device="cuda", generator=gen) * 6
        d = 700 + 180 * torch.sin(xx) * torch.cos(yy) + 3 * torch.randn((h, w), device="cuda", generator=gen)
        d = d.round().clamp(300, 1050).to(torch.int32)
        d[torch.rand((h, w), device="cuda", generator=gen) < 0.05] = 2047
        s["disparity"] = d.to(torch.int16)
        cal = synth.calib_block_np(w, h)
        cal[61], cal[42] = 3.330949516e-3, -3.07110156e-6  # a Kinect's 1 / z in 1 / mm: c0 + c1 disparity
        s["calib"] = cal
        oh, ow = (h // 2, w // 2) if case["half"] else (h, w)
        s["depth"] = torch.empty((oh, ow), dtype=torch.float32, device="cuda")
        s["depth16"] = torch.empty((oh, ow), dtype=torch.int16, device="cuda")
        s["buffers"] = _Frames(s["disparity"]), _Frames(s["depth"]), _Frames(s["depth16"])
    elif kind == "pair":
        w, h = case["width"], case["height"]
        pairs, _, s["frames"] = _frame_pairs(seed, [(w, h)], 1.5, 25.0)
        s["pair"] = pairs[0]
        s["tracker"] = PhotoTracker(w, h, pairs[0]["calib"], mode=MODES[case["mode"]], n_select=case["points"], lam=0.5,
                                    iters=ITERS)
    elif kind == "sequence":
        w, h = case["width"], case["height"]
        s["gray"], s["depth"], _ = _sequence(seed, case["frames"], w, h, 1.5, 20.0)
        s["tracker"] = PhotoTracker(w, h, synth.calib_block_np(w, h), mode=MODES[case["mode"]], n_select=case["points"],
                                    lam=0.5, iters=ITERS)
    elif kind == "pipeline":
        w, h = case["width"], case["height"]
        s["gray"], s["depth"], _ = _sequence(seed, case["frames"], w, h, 2.0, 20.0)
        s["buffers"] = _Frames(s["gray"]), _Frames(s["depth"])
        s["net"] = PoseNet.load(max_batch=64)
        s["engine"] = SequenceTracker(w, h, synth.calib_block_np(w, h), net=s["net"], n_select=case["points"],
                                      reloc_points=min(8192, case["points"]))
    elif kind in ("batch", "learned"):
        n, w, h = case["pairs"], case["width"], case["height"]
        sizes = [(w, h)] * n if w else [MIXED[k] for k in np.random.default_rng(seed).integers(0, len(MIXED), n)]
        large = kind == "learned"
        pairs, _, s["frames"] = _frame_pairs(seed, sizes, 10.0 if large else 1.5, 150.0 if large else 25.0)
        mode = MODES[case["mode"]] if kind == "batch" else PHOTOMETRIC
        s["batch"] = BatchTracker(n, max(x for x, _ in sizes), max(y for _, y in sizes), mode=mode,
                                  n_select=case["points"], lam=0.5, iters=ITERS)
        s["pairs"] = s["batch"].prepare(pairs)
        if large:
            s["net"] = PoseNet.load(max_batch=n)
    elif kind in ("forward", "gradient"):
        n = case["pairs"]
        if kind == "forward":
            net = s["net"] = PoseNet.load(max_batch=n)
        else:  # a training run starts from these
            net = s["net"] = PoseNet(max_batch=n)
            net.set_params(init_params(net.cfg, seed=1))
        s["x"], motions, s["frames"] = _net_inputs(seed, n, net)
        if kind == "forward":
            s["out"] = torch.empty((n, 6), dtype=torch.float32, device="cuda")
        else:
            y = pose_to_target(net.cfg, np.linalg.inv(motions))
            s["y"] = torch.from_numpy(y).cuda()
            s["w"] = torch.ones(n, dtype=torch.float32, device="cuda")
    else:
        w, h, res = case["width"], case["height"], case["resolution"]
        _, s["depth"], poses = _sequence(seed, 4, w, h, 1.0, 15.0, noise=0.0)
        fx, fy, cx, cy = synth.pinhole(w, h)
        s["K"] = np.array([-fx / w, 0, cx / w, 0, fy / h, cy / h, 0, 0, 1], np.float32)
        s["poses"] = [np.ascontiguousarray(p, np.float32).ravel() for p in poses]
        g = s["grid"] = VoxelGrid(default_params(resolution=res, width=w, height=h))
        for k in range(3):  # the model holds the frames before this one
            check(lib().rt_tsdf_set_depth_u16(g.h, s["depth"][k].data_ptr()), "rt_tsdf_set_depth_u16")
            g.update(s["poses"][k], s["K"])
        g.synchronize()
        s["maps"] = [torch.zeros((h, w, 4), dtype=torch.float32, device="cuda") for _ in range(3)]
        s["voxels"] = torch.as_tensor(_Voxels(g), device="cuda")
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------ run
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "disparity":
        h, w = s["disparity"].shape
        d, z, z16 = s["buffers"]
        disparity_to_depth((d, h, w), s["calib"], xy_offset=True, half=case["half"], out=z)
        depth_mm_to_u16(z, s["depth"].numel(), z16)
        return {"mm": s["depth"], "u16": s["depth16"]}
    if kind == "pair":
        t, p = s["tracker"], s["pair"]
        t.set_reference_points(p["ref_gray"], p["ref_depth"], mode=MODES[case["mode"]], lam=0.5, force=True,
                               on_device=True)
        t.set_current_image(p["cur_gray"], p["cur_depth"], on_device=True)
        t.track()
        return {"pose": t.get_relative_pose()}
    if kind == "sequence":
        return {"poses": s["tracker"].track_sequence(s["gray"].data_ptr(), s["depth"].data_ptr(), case["frames"],
                                                     case["interval"], case["fuse"])}
    if kind == "pipeline":
        poses, stats = s["engine"].run(s["buffers"][0], s["buffers"][1], case["frames"])
        return {"poses": poses, "rms": np.array([t[1] for t in stats["trace"]], np.float32),
                "keyframe": np.array([t[0] for t in stats["trace"]], np.int32)}
    if kind == "batch":
        Trel, T, rms, status = s["batch"].track(s["pairs"])
        return {"Trel": Trel, "T": T, "rms": rms, "status": status}
    if kind == "learned":
        b = s["batch"]
        b.prepare_only(s["pairs"])
        b.propose(s["net"])
        Trel, T, rms, status = b.retrack(None, case["pairs"])
        return {"Trel": Trel, "T": T, "rms": rms, "status": status}
    if kind == "forward":
        s["net"].forward(case["pairs"], s["x"].data_ptr(), s["out"].data_ptr())
        return {"out": s["out"]}
    if kind == "gradient":
        loss, out, grad = s["net"].loss_grad(case["pairs"], s["x"].data_ptr(), s["y"].data_ptr(), s["w"].data_ptr())
        return {"loss": np.float32(loss), "out": out, "grad": grad}
    g, L = s["grid"], lib()
    fp = ctypes.POINTER(ctypes.c_float)
    T, K = s["poses"][3].ctypes.data_as(fp), s["K"].ctypes.data_as(fp)
    check(L.rt_tsdf_set_depth_u16(g.h, s["depth"][3].data_ptr()), "rt_tsdf_set_depth_u16")
    check(L.rt_tsdf_update(g.h, T, K), "rt_tsdf_update")
    check(L.rt_tsdf_raycast(g.h, T, K, 1, *(m.data_ptr() for m in s["maps"])), "rt_tsdf_raycast")
    return {"voxels": s["voxels"], "xyz": s["maps"][0], "normals": s["maps"][1], "shade": s["maps"][2]}


# ------------------------------------------------------------------ work
def _tracking_flops(width, height, mode, points):
    """About 120 operations per keyframe pixel of preparation; per iteration
    about 150 per photometric point and 130 per pixel of the geometric level."""
    levels = 4 if width == 640 else 3
    f = 120 * width * height
    for k in range(levels):
        layer = levels - 1 - k
        if mode != "geometric":
            f += ITERS[k] * 150 * points
        if mode != "photometric":
            f += ITERS[k] * 130 * (width >> layer) * (height >> layer)
    return f


def work(case):
    kind = case["kind"]
    if kind == "disparity":
        n = case["width"] * case["height"]
        o = n // 4 if case["half"] else n
        return {"bytes": 2 * n + 6 * o, "flops": 8 * o}
    if kind == "pair":
        n = case["width"] * case["height"]
        return {"bytes": 6 * n + 64, "flops": _tracking_flops(case["width"], case["height"], case["mode"], case["points"])}
    if kind in ("sequence", "pipeline"):
        n, f = case["width"] * case["height"], case["frames"]
        per = _tracking_flops(case["width"], case["height"], case.get("mode", "bi-objective"), case["points"])
        if kind == "pipeline":
            per += 2 * NET_MACS
        return {"bytes": 3 * n * f + 128 * f, "flops": per * f}
    if kind in ("batch", "learned"):
        sizes = [(case["width"], case["height"])] if case["width"] else list(MIXED)
        px = sum(w * h for w, h in sizes) / len(sizes)
        fl = sum(_tracking_flops(w, h, case.get("mode", "photometric"), case["points"]) for w, h in sizes) / len(sizes)
        if kind == "learned":
            fl += 2 * NET_MACS
        return {"bytes": case["pairs"] * (6 * px + 264), "flops": case["pairs"] * fl}
    if kind in ("forward", "gradient"):
        n = case["pairs"]
        b = n * (60 * 80 * 4 * 2 + 24) + 2 * NET_PARAMS
        if kind == "forward":
            return {"bytes": b, "flops": 2 * NET_MACS * n}
        return {"bytes": b + 4 * NET_PARAMS + 28 * n, "flops": 6 * NET_MACS * n}
    # about a quarter of the grid's voxels lie in the view before the surface: read and written;
    # the view's maps are written, its depth read
    v, n = case["resolution"] ** 3, case["width"] * case["height"]
    return {"bytes": 16 * v // 4 + 50 * n, "flops": 30 * v + 20 * case["resolution"] * n}


# ------------------------------------------------------------------ exact
def _exact_disparity(case, s):
    d = s["disparity"].cpu().numpy().astype(np.int64)
    cal = s["calib"]
    c0, c1, mn, mx = (float(cal[k]) for k in (61, 42, 62, 63))
    h, w = d.shape
    oh, ow = s["depth"].shape
    step = 2 if case["half"] else 1
    sx, sy = step * np.arange(ow) - 4, step * np.arange(oh) - 3
    inside = ((sx >= 0) & (sx < w - 1))[None, :] & ((sy >= 0) & (sy < h - 1))[:, None]
    X, Y = np.clip(sx, 0, w - 2)[None, :], np.clip(sy, 0, h - 2)[:, None]
    taps = [d[Y, X]] + ([d[Y, X + 1], d[Y + 1, X], d[Y + 1, X + 1]] if case["half"] else [])
    m = np.minimum.reduce(taps)
    valid = inside & (np.maximum.reduce(taps) < 2047) & (np.arange(oh) < 4 * (oh // 4))[:, None]
    z = np.abs(1.0 / (c0 + c1 * m))
    return np.where(valid & (z >= mn) & (z <= mx), z, 0.0)


def _exact_net(x, params, cfg, y=None, w=None):
    """The network in float64 from its float32 parameters, and the gradients
    of its loss in the flat parameter layout."""
    dev = x.device
    p = torch.from_numpy(np.asarray(params, np.float64)).to(dev).requires_grad_(y is not None)
    ch = list(cfg.channels)
    total = torch.zeros(len(params), dtype=torch.float64, device=dev)
    outs, loss = [], 0.0
    wsum = max(1.0, float(w.double().sum())) if w is not None else 1.0
    for a in range(0, len(x), 32):  # images at a time: the columns of a layer are its input nine times over
        t = x[a:a + 32].double()
        o = 0
        for l in range(6):
            ci, co = ch[l], ch[l + 1]
            W = p[o:o + co * 9 * ci].view(co, 9 * ci)
            o += co * 9 * ci
            b = p[o:o + co]
            o += co
            n, hh, ww, _ = t.shape
            oh, ow = (hh + 1) // 2, (ww + 1) // 2
            tp = torch.nn.functional.pad(t, (0, 0, 1, 1, 1, 1))
            cols = torch.cat([tp[:, ky:ky + 2 * oh - 1:2, kx:kx + 2 * ow - 1:2, :] for ky in range(3) for kx in range(3)],
                             dim=3)
            t = torch.relu(cols.reshape(-1, 9 * ci) @ W.t() + b).view(n, oh, ow, co)
        f = t.mean(dim=(1, 2))
        r = f @ p[o:o + 6 * ch[6]].view(6, ch[6]).t() + p[o + 6 * ch[6]:o + 6 * ch[6] + 6]
        outs.append(r.detach())
        if y is not None:
            part = (w[a:a + 32, None].double() * (r - y[a:a + 32].double()) ** 2).sum() / wsum
            total += torch.autograd.grad(part, p)[0]
            loss += float(part)
    return torch.cat(outs), loss, total


def exact(case, seed):
    kind = case["kind"]
    if kind == "disparity":
        # the rounded 16-bit map has no value of its own in 64 bits: it is whole numbers
        return {"mm": _exact_disparity(case, prepare(case, seed)), "u16": None}
    if kind in ("forward", "gradient"):
        s = prepare(case, seed)
        params = s["net"].get_params()
        if kind == "forward":
            with torch.no_grad():
                return {"out": _exact_net(s["x"], params, s["net"].cfg)[0]}
        out, loss, grad = _exact_net(s["x"], params, s["net"].cfg, s["y"], s["w"])
        return {"loss": np.float64(loss), "out": out.cpu().numpy(), "grad": grad.cpu().numpy()}
    # The trackers settle by rounded decisions (selected points, gradient and median bins, keyframe
    # switches), the voxel grid by thresholds per voxel: in 64 bits these take other ways, and the
    # results are those of another selection.
    return None
