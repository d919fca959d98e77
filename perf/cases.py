"""The work that users of this framework have it do, as timed cases.

Kinds of case, each called as a program calls it:
  paint    one frame of an interactive view: HIPRaycaster.Paint() into host memory
  views    frames of an orbit that stay on the device for a consumer there:
           PaintViews(download=False, stats=False) and the frame pointer
  batch    a render service: many requests over shared volumes, one RenderBatch.Render()
  leap     one pass of the ray-guided traversal: HIPRaycaster.LeapRender()
  convert  a raw volume in host memory to the bricks of every level: LoadVolume, GetPool
  rebrick  a resident volume bricked anew on the device, its gradient maximum, a first frame
  train    the step network trained on recorded chunks: StepNet.train()
"""
import ctypes as C
import math

import numpy as np
import torch

from tuvok_amd import (DISPATCH_GROUPS, DISPATCH_QUEUES, GEN_BLOBS, GEN_ELLIPSOID_SDF, GEN_FBM_SHELLS, GEN_PHANTOM,
                       RM_1DTRANS, RM_2DTRANS, RM_ISOSURFACE, HIPRaycaster, RenderBatch, _abi)
from tuvok_amd.stepnet import StepNet, labels, split_samples

ERT = 2.0 ** -11
GENERATORS = {"blobs": GEN_BLOBS, "fbm": GEN_FBM_SHELLS, "sdf": GEN_ELLIPSOID_SDF, "phantom": GEN_PHANTOM}
MODES = {"1d": RM_1DTRANS, "2d": RM_2DTRANS, "iso": RM_ISOSURFACE}


# ---- the cases ---------------------------------------------------------------------

def _paint(dims, bits, brick, mode, lit, w, h, srm=1.0, ert=0.0):
    return dict(kind="paint", x=dims[0], y=dims[1], z=dims[2], bits=bits, brick=brick, mode=mode, lit=lit, w=w, h=h,
                srm=srm, ert=ert)


def _views(gen, edge, bits, brick, mode, lit, w, h, views, srm=1.0, ert=ERT, step="fixed"):
    return dict(kind="views", gen=gen, edge=edge, bits=bits, brick=brick, mode=mode, lit=lit, w=w, h=h, views=views,
                srm=srm, ert=ert, step=step)


def listed():
    return [
        # the smallest frame: a thumbnail of a small volume, where launches and copies count
        dict(_paint((64, 64, 64), 8, 18, "1d", False, 64, 64), name="paint_64_u8_1d"),
        # an interactive window on a 256^3 volume with a 1D transfer function
        dict(_paint((256, 256, 256), 8, 66, "1d", False, 512, 512), name="paint_512_u8_1d"),
        # a ragged volume and window, shaded 2D transfer function, the reference's exact termination
        dict(_paint((253, 190, 141), 16, 66, "2d", True, 641, 479), name="paint_odd_u16_2d_lit"),
        # the headline orbit: 1024^3 uint16, shaded 2D transfer function, 16 frames of 1920x1080
        dict(_views("fbm", 1024, 16, 130, "2d", True, 1920, 1080, 16), name="orbit_1024_u16_2d_lit"),
        # a sparse scan-like volume, shaded 1D transfer function at the 0.25-voxel step, 4 frames
        dict(_views("phantom", 1024, 16, 130, "1d", True, 1920, 1080, 4, srm=2.0), name="orbit_1024_u16_1d_lit"),
        # the same with the learned step proposal
        dict(_views("phantom", 1024, 16, 130, "1d", True, 1920, 1080, 4, srm=2.0, step="learned"),
             name="orbit_1024_u16_learned"),
        # the isosurface of a large distance field, one frame
        dict(_views("sdf", 2048, 8, 130, "iso", True, 1920, 1080, 1), name="iso_2048_u8"),
        # a service's batch: requests of uneven sizes over three uint8 volumes, 1D transfer functions
        dict(kind="batch", edge=1024, requests=24, min_px=256, max_px=2048, mode="1d", lit=False, tile_w=8,
             name="batch_24_u8_1d"),
        # one ray-guided pass over every level of a 1024^3 volume, 1920x1080
        dict(kind="leap", gen="fbm", edge=1024, bits=16, brick=130, mode="2d", lit=True, w=1920, h=1080,
             name="leap_1024_u16_2d_lit"),
        # a raw scan converted to bricks with every level, ragged sizes
        dict(kind="convert", x=301, y=277, z=190, bits=16, brick=66, name="convert_u16"),
        # a new brick size and pyramid for a resident volume, and its first frame
        dict(kind="rebrick", gen="fbm", edge=1024, bits=16, brick=130, w=1024, h=768, name="rebrick_1024_u16"),
        # training of the step network on recorded chunks
        dict(kind="train", n=100000, epochs=2, batch=4096, name="train_100k"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["paint", "paint", "paint", "views", "views", "views", "batch", "leap", "convert", "rebrick",
                       "train"])
    bits = rng.choice([8, 16])
    if kind == "paint":
        dims = [_log(rng, 40, 320) for _ in range(3)]
        return _paint(dims, bits, rng.choice([18, 34, 66, 130]) if max(dims) <= 128 else rng.choice([66, 130]),
                      rng.choice(["1d", "1d", "2d"]), rng.random() < 0.5, _log(rng, 48, 1280), _log(rng, 48, 800),
                      srm=rng.choice([1.0, 1.0, 2.0]), ert=rng.choice([0.0, ERT]))
    if kind == "views":
        mode = rng.choice(["1d", "2d", "iso"])
        gen = "sdf" if mode == "iso" else rng.choice(["fbm", "blobs"] if bits == 8 else ["fbm", "phantom"])
        edge = _log(rng, 128, 1024)
        return _views(gen, edge, 8 if gen == "sdf" else bits, 66 if edge < 400 else 130, mode, rng.random() < 0.5,
                      _log(rng, 256, 1920), _log(rng, 256, 1080), rng.choice([1, 1, 2, 4]), srm=rng.choice([1.0, 1.0, 2.0]))
    if kind == "batch":
        return dict(kind="batch", edge=_log(rng, 256, 1024), requests=rng.randint(2, 24), min_px=64,
                    max_px=_log(rng, 256, 1536), mode=rng.choice(["1d", "1d", "iso"]), lit=rng.random() < 0.5,
                    tile_w=rng.choice([8, 8, 4, 16]))
    if kind == "leap":
        return dict(kind="leap", gen="fbm", edge=rng.choice([256, 512, 1024]), bits=bits, brick=rng.choice([66, 130]),
                    mode=rng.choice(["1d", "2d"]), lit=rng.random() < 0.5, w=_log(rng, 256, 1920), h=_log(rng, 256, 1080))
    if kind == "convert":
        return dict(kind="convert", x=_log(rng, 40, 400), y=_log(rng, 40, 400), z=_log(rng, 40, 400), bits=bits,
                    brick=rng.choice([34, 66, 130]))
    if kind == "rebrick":
        return dict(kind="rebrick", gen="fbm", edge=_log(rng, 128, 1024), bits=bits, brick=rng.choice([66, 130, 258]),
                    w=_log(rng, 256, 1024), h=_log(rng, 256, 768))
    return dict(kind="train", n=_log(rng, 4096, 200000), epochs=rng.choice([1, 2]), batch=rng.choice([1024, 4096]))


# ---- inputs ---------------------------------------------------------------------------

def _volume(case, seed):
    """A scan-like volume (z, y, x) of whole numbers: Gaussian blobs, a hollow shell and a little noise."""
    X, Y, Z = case["x"], case["y"], case["z"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    r = np.random.default_rng(seed)
    gx, gy, gz = ((torch.arange(n, dtype=torch.float64, device=dev) + 0.5) / n for n in (X, Y, Z))
    v = torch.zeros((Z, Y, X), dtype=torch.float64, device=dev)
    for _ in range(10):
        c, s, a = r.uniform(0.2, 0.8, 3), r.uniform(0.04, 0.13), r.uniform(0.3, 0.8)
        e = [torch.exp(-((g - q) ** 2) / (2 * s * s)) for g, q in zip((gx, gy, gz), c)]
        v += a * e[2][:, None, None] * e[1][None, :, None] * e[0][None, None, :]
    c, rad = r.uniform(0.4, 0.6, 3), r.uniform(0.2, 0.35)
    d = (((gz - c[2]) ** 2)[:, None, None] + ((gy - c[1]) ** 2)[None, :, None] + ((gx - c[0]) ** 2)[None, None, :]).sqrt()
    v = torch.where((d - rad).abs() < 1.5 / max(X, Y, Z), torch.full_like(v, 0.9), v)
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))
    v += 0.01 * torch.rand(v.shape, generator=g, device=dev, dtype=torch.float64)
    top = 255 if case["bits"] == 8 else 65535
    return (v.clamp(0, 1) * top).floor().to(torch.int32)


def _host(vol, bits):
    return vol.cpu().numpy().astype(np.uint8 if bits == 8 else np.uint16)


def _table_1d(seed, n=256):
    """A 1D transfer function: transparent below a threshold, then a ramp between two colours."""
    r = np.random.default_rng([seed, 1])
    lo, top, c0, c1 = int(r.integers(25, 90)), r.uniform(0.2, 0.8), r.uniform(0, 1, 3), r.uniform(0, 1, 3)
    i = np.arange(n)
    t = np.zeros((n, 4))
    t[:, :3] = c0 + (c1 - c0) * (i / (n - 1))[:, None]
    t[:, 3] = np.where(i < lo, 0.0, top * (i - lo) / (n - 1 - lo))
    return (np.clip(t, 0, 1) * 255).astype(np.uint8)


def _table_2d(seed, n=256):
    """A 2D transfer function of four lobes over value and gradient (rows from steep to flat)."""
    r = np.random.default_rng([seed, 2])
    x, y = np.meshgrid((np.arange(n) + 0.5) / n, (np.arange(n) + 0.5) / n)
    rgb, a = np.zeros((n, n, 3)), np.zeros((n, n))
    for vc, gc, vs, gs, top in ((0.30, 0.95, 0.05, 0.05, 0.05), (0.55, 0.85, 0.06, 0.10, 0.10),
                                (0.75, 0.70, 0.05, 0.15, 0.30), (0.915, 0.90, 0.02, 0.12, 0.90)):
        w = top * np.exp(-0.5 * (((x - vc - r.uniform(-0.02, 0.02)) / vs) ** 2 + ((y - gc) / gs) ** 2))
        rgb += w[..., None] * r.uniform(0.3, 1.0, 3)
        a += w
    rgb = np.where(a[..., None] > 0, rgb / np.maximum(a[..., None], 1e-12), 0)
    return (np.clip(np.concatenate([rgb, a[..., None]], -1), 0, 1) * 255).astype(np.uint8)


def _angles(seed, n):
    """An orbit about the vertical axis from a random start."""
    return np.random.default_rng([seed, 3]).uniform(0, 2 * math.pi) + 2 * math.pi * np.arange(n) / n


def _rotation(a):
    c, s = np.float32(math.cos(a)), np.float32(math.sin(a))
    return np.array([[c, 0, -s, 0], [0, 1, 0, 0], [s, 0, c, 0], [0, 0, 0, 1]], np.float32)


def _dtype(bits):
    return np.uint8 if bits == 8 else np.uint16


def _look(ren, case, seed, eye=2.0):
    """Transfer function, mode and camera of a renderer whose dataset is set."""
    if case["mode"] == "1d":
        ren.Set1DTrans(_table_1d(seed))
    elif case["mode"] == "2d":
        ren.Set2DTrans(_table_2d(seed))
        ren.SetGradientScale(1.0 / ren.MaxGradientMagnitude())
    ren.SetRendermode(MODES[case["mode"]])
    ren.SetUseLighting(case["lit"])
    if case["mode"] == "iso":
        ren.SetIsoValue(128.0)
        ren.SetRefineSteps(4)
    ren.SetSampleRateModifier(case.get("srm", 1.0))
    ren.SetEarlyRayTermination(case.get("ert", 0.0))
    ren.SetViewParameters(45.0, 0.01, 1000.0)
    ren.SetViewPosition((0.0, 0.0, eye))
    ren.Resize(case["w"], case["h"])


def _proposal(ren, rots, seed):
    """A step network trained on recorded chunks of these views, always in the same order."""
    rec = ren.GenerateSegments(rots, 50000, seed=seed, fit=True)[:, :42]
    rec = np.ascontiguousarray(rec)
    rec = rec[np.argsort(rec.view("V168").reshape(-1), kind="stable")]
    net = StepNet(0, seed=seed)
    net.set_data(split_samples(rec)[0], labels(rec, 0.25 / 255, 0.125 / 255))
    net.train(epochs=4, seed=seed)
    return net


class _DeviceFrames:
    """Frames that a renderer left on the device, for torch to wrap without a copy: the tensor holds this object, and
    with it the renderer that owns the memory."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f4", data=(int(ptr), False), version=2)


def _frames(call, owner, shape, *more):
    p = C.c_void_p()
    if call(owner._h, *more, C.byref(p)) != 0:
        raise RuntimeError("no frame pointer")
    return torch.as_tensor(_DeviceFrames(owner, p.value, shape), device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "paint":
        ren = HIPRaycaster(0)
        ren.LoadVolume(_host(_volume(case, seed), case["bits"]), (case["brick"],) * 3, 1, max_lods=1)
        _look(ren, case, seed)
        ren.SetRotation(_rotation(_angles(seed, 1)[0]))
        return dict(case=case, ren=ren)
    if kind == "views":
        ren = HIPRaycaster(0)
        ren.GenerateVolume(GENERATORS[case["gen"]], seed, _dtype(case["bits"]), (case["edge"],) * 3, (case["brick"],) * 3,
                           1, max_lods=1)
        _look(ren, case, seed)
        net = None
        if case["step"] == "learned":
            ren.Resize(240, 135)
            net = _proposal(ren, [_rotation(a) for a in _angles(seed + 1, 4)], seed)
            ren.Resize(case["w"], case["h"])
            ren.SetStepProposal(net, margin=1.0, skip_threshold=0.999, fallback_bound=0.01)
        if case["gen"] in ("phantom", "sdf"):
            # what the dispatch tuner picks for sparse volumes
            ren.SetDispatchOrder(DISPATCH_GROUPS | DISPATCH_QUEUES)
        return dict(case=case, ren=ren, net=net, rots=[_rotation(a) for a in _angles(seed, case["views"])])
    if kind == "batch":
        r = np.random.default_rng([seed, 4])
        owners = []
        for gen, edge in (("blobs", max(64, case["edge"] // 4)), ("sdf", max(96, case["edge"] // 2)), ("sdf", case["edge"])):
            ren = HIPRaycaster(0)
            ren.GenerateVolume(GENERATORS[gen], int(r.integers(1 << 30)), np.uint8, (edge,) * 3,
                               (130 if edge >= 512 else 66,) * 3, 1, max_lods=1)
            owners.append(ren)
        batch, rens, sizes = RenderBatch(0), [], []
        batch.SetTuning(case["tile_w"], 64 // case["tile_w"])
        q = np.random.default_rng([case["requests"], case["max_px"]])   # the requests' sizes and volumes
        for k in range(case["requests"]):
            w, h = (int(round(math.exp(q.uniform(math.log(case["min_px"]), math.log(case["max_px"]))))) for _ in range(2))
            ren = HIPRaycaster(0)
            ren.ShareDataset(owners[int(q.integers(len(owners)))])
            _look(ren, dict(case, w=w, h=h, ert=ERT), int(r.integers(1 << 30)))
            rot = _rotation(r.uniform(0, 2 * math.pi))
            batch.Add(ren, rot, w, h)
            rens.append(ren)
            sizes.append((w, h))
        return dict(case=case, batch=batch, rens=rens, owners=owners, sizes=sizes)
    if kind == "leap":
        ren = HIPRaycaster(0)
        ren.GenerateVolume(GENERATORS[case["gen"]], seed, _dtype(case["bits"]), (case["edge"],) * 3, (case["brick"],) * 3, 1)
        _look(ren, case, seed)
        ren.SetRotation(_rotation(_angles(seed, 1)[0]))
        ren.LeapSetResident(None)
        return dict(case=case, ren=ren)
    if kind == "convert":
        return dict(case=case, ren=HIPRaycaster(0), vol=_host(_volume(case, seed), case["bits"]))
    if kind == "rebrick":
        ren = HIPRaycaster(0)
        ren.GenerateVolume(GENERATORS[case["gen"]], seed, _dtype(case["bits"]), (case["edge"],) * 3, (66,) * 3, 1,
                           max_lods=1, keep_linear=True)
        _look(ren, dict(case, mode="2d", lit=True, ert=ERT), seed, eye=2.5)
        ren.SetLOD(-1)
        return dict(case=case, ren=ren, rots=[_rotation(_angles(seed, 1)[0])])
    r = np.random.default_rng([seed, 5])
    n = case["n"]
    feat = r.random((n, 24), np.float32)
    feat[:, 9:11] = r.integers(0, 2, (n, 2))
    feat[:, 23] = 1.0
    k = np.clip(np.floor(4 * (1 - feat[:, 19] * feat[:, 5])), 0, 3)
    tgt = np.stack([k / 3, feat[:, 19] < 0.2, np.ones(n)], axis=1).astype(np.float32)
    net = StepNet(0, seed=seed)
    net.set_data(feat, tgt)
    return dict(case=case, net=net, start=net.get_params())


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "paint":
        return state["ren"].Paint()
    if kind == "views":
        ren = state["ren"]
        ren.PaintViews(state["rots"], download=False, stats=False)
        return _frames(_abi.load().tvk_frame_device_ptr, ren, (case["views"], case["h"], case["w"], 4))
    if kind == "batch":
        b = state["batch"]
        b.Render()
        call = _abi.load().tvk_batch_frame_device_ptr
        return [_frames(call, b, (h, w, 4), i) for i, (w, h) in enumerate(state["sizes"])]
    if kind == "leap":
        return state["ren"].LeapRender(first=True)[0]
    if kind == "convert":
        ren = state["ren"]
        ren.LoadVolume(state["vol"], (case["brick"],) * 3, 1)
        return [ren.GetPool(), ren.MaxGradientMagnitude()]
    if kind == "rebrick":
        ren = state["ren"]
        ren.Rebrick((case["brick"],) * 3, 1, max_lods=0)
        g = ren.MaxGradientMagnitude()
        ren.SetGradientScale(1.0 / g)
        ren.PaintViews(state["rots"], download=False, stats=False)
        return [g, _frames(_abi.load().tvk_frame_device_ptr, ren, (1, case["h"], case["w"], 4))]
    net = state["net"]
    net.set_params(state["start"])   # every pass trains from the same start
    losses = net.train(epochs=case["epochs"], batch=case["batch"], seed=7)
    return [net.get_params(), losses]


def work(case):
    """Bytes: the volume's voxels read once (for conversions the bricks of all levels written too) and each frame
    written once.  Operations: the products of the network; a march's depend on where its rays end and are left out."""
    kind = case["kind"]
    bpv = case.get("bits", 8) // 8
    if kind == "train":
        per_sample = 3 * 2 * (24 * 64 + 64 * 64 + 64 * 2)
        return {"bytes": case["n"] * 27 * 4 * case["epochs"], "flops": per_sample * case["n"] * case["epochs"]}
    if kind == "convert":
        vox = case["x"] * case["y"] * case["z"]
        stored = (case["brick"] / (case["brick"] - 2)) ** 3
        return {"bytes": int(vox * bpv * (1 + stored * 8 / 7)), "flops": 0}
    if kind == "batch":
        mean = (case["max_px"] - case["min_px"]) / math.log(case["max_px"] / case["min_px"])
        vox = sum(e ** 3 for e in (max(64, case["edge"] // 4), max(96, case["edge"] // 2), case["edge"]))
        return {"bytes": int(vox + case["requests"] * mean * mean * 16), "flops": 0}
    pixels = case["w"] * case["h"] * case.get("views", 1)
    vox = case["x"] * case["y"] * case["z"] if kind == "paint" else case["edge"] ** 3
    if kind == "rebrick":
        stored = (case["brick"] / (case["brick"] - 2)) ** 3
        return {"bytes": int(vox * bpv * (1 + stored * 8 / 7) + pixels * 16), "flops": 0}
    return {"bytes": vox * bpv + pixels * 16, "flops": 0}


# ---- the frame of a paint case in 64 bits -----------------------------------------------

def _bricks(vol, b):
    """(first voxel, core size, stored voxels with the zero border) of every brick, overlap 1."""
    core = b - 2
    p = torch.nn.functional.pad(vol, (1,) * 6)
    for z in range(0, vol.shape[0], core):
        for y in range(0, vol.shape[1], core):
            for x in range(0, vol.shape[2], core):
                n = [min(core, s - o) for s, o in zip(vol.shape[::-1], (x, y, z))]
                yield (x, y, z), n, p[z:z + n[2] + 2, y:y + n[1] + 2, x:x + n[0] + 2]


def _lerp(brick, u):
    """Trilinear value at texel positions u (..., 3), 0 outside the brick (brick: one more ring of zeros)."""
    n = torch.tensor(brick.shape[::-1], device=u.device, dtype=u.dtype) - 2
    u = torch.minimum(torch.clamp(u, min=-0.5), n - 0.5)
    i = torch.floor(u)
    f = u - i
    i = i.long() + 1
    flat = brick.reshape(-1)
    sx, sy = brick.shape[2], brick.shape[2] * brick.shape[1]
    base = i[..., 0] + i[..., 1] * sx + i[..., 2] * sy
    out = 0
    for k in range(8):
        w = 1
        for a in range(3):
            w = w * (f[..., a] if (k >> a) & 1 else 1 - f[..., a])
        out = out + w * flat[base + (k & 1) + ((k >> 1) & 1) * sx + (k >> 2) * sy]
    return out


def exact(case, seed):
    if case["kind"] == "convert":   # the pool holds whole numbers; the gradient maximum of the brick cores
        v = torch.nn.functional.pad(_volume(case, seed).to(torch.float64), (1,) * 6)
        g2 = ((v[1:-1, 1:-1, :-2] - v[1:-1, 1:-1, 2:]) ** 2 + (v[1:-1, :-2, 1:-1] - v[1:-1, 2:, 1:-1]) ** 2 +
              (v[:-2, 1:-1, 1:-1] - v[2:, 1:-1, 1:-1]) ** 2)
        return [None, float(g2.max().sqrt()) / (2 * (255 if case["bits"] == 8 else 65535))]
    if case["kind"] != "paint" or case["x"] * case["y"] * case["z"] * case["srm"] > 2 ** 24 * 1.2:
        return None   # the others hold whole numbers, or would take too long
    f8 = dict(dtype=torch.float64, device="cuda" if torch.cuda.is_available() else "cpu")
    vol = _volume(case, seed)
    W, H, srm, ert, lit = case["w"], case["h"], case["srm"], case["ert"], case["lit"]
    top = 255.0 if case["bits"] == 8 else 65535.0
    dims = torch.tensor([case["x"], case["y"], case["z"]], **f8)
    edge = float(dims.max())
    data = torch.nn.functional.pad(vol.to(torch.float64), (1,) * 6)
    g = [(data[1:-1, 1:-1, :-2] - data[1:-1, 1:-1, 2:]), (data[1:-1, :-2, 1:-1] - data[1:-1, 2:, 1:-1]),
         (data[:-2, 1:-1, 1:-1] - data[2:, 1:-1, 1:-1])]
    gscale = 2 * top / float((g[0] ** 2 + g[1] ** 2 + g[2] ** 2).sqrt().max())
    del data, g
    high = float(vol.max())
    two = case["mode"] == "2d"
    table = torch.tensor((_table_2d if two else _table_1d)(seed), **f8) / 255
    opaque = table[..., 3].amax(0) if two else table[:, 3]
    some = torch.nonzero(opaque).reshape(-1)
    unit = high / (len(opaque) - 1)
    first, last = int(some[0]) * unit, int(some[-1]) * unit
    # eye space: the eye at the origin, the volume turned and moved to distance 2
    mv = torch.tensor(_rotation(_angles(seed, 1)[0]), **f8)
    mv[3, 2] = -2.0
    inv = torch.linalg.inv(mv)
    tan = math.tan(math.radians(45.0) / 2)
    px = ((torch.arange(W, **f8) + 0.5) * 2 / W - 1) * tan * W / H * 0.01
    py = ((torch.arange(H, **f8) + 0.5) * 2 / H - 1) * tan * 0.01
    d = torch.stack([px.expand(H, W), py[:, None].expand(H, W), torch.full((H, W), -0.01, **f8)], -1).reshape(-1, 3)
    om, dm = inv[3, :3], d @ inv[:3, :3]
    amb, light = 0.1, torch.tensor([0.0, 0.0, -1.0], **f8)
    todo = []
    for first_voxel, n, stored in _bricks(vol, case["brick"]):
        lo = torch.tensor(first_voxel, **f8) / edge - dims / edge / 2
        size = torch.tensor(n, **f8) / edge
        if not (last >= float(stored.min()) and first <= float(stored.max())):
            continue
        mid = lo + size / 2
        corner = torch.tensor([[sx, sy, sz] for sx in (-1, 1) for sy in (-1, 1) for sz in (-1, 1)], **f8)
        eye = (mid + corner * size * 0.4999) @ mv[:3, :3] + mv[3, :3]
        todo.append((float(eye.norm(dim=1).min()), lo, size, stored))
    out = torch.zeros((H * W, 4), **f8)
    for _, lo, size, stored in sorted(todo, key=lambda t: t[0]):
        t0, t1 = (lo - om) / dm, (lo + size - om) / dm
        tn, tf = torch.minimum(t0, t1).amax(1), torch.maximum(t0, t1).amin(1)
        te = tn.clamp(min=1.0)
        live = torch.nonzero((tf > te) & ~((ert > 0) & (1 - out[:, 3] < ert))).reshape(-1)
        nv = torch.tensor(stored.shape[::-1], **f8)
        step = float((size / nv).min()) * 0.5 / srm
        brick = torch.nn.functional.pad(stored.to(torch.float64), (1,) * 6) / top
        for part in torch.split(live, 1 << 16):
            entry = (d[part] * te[part, None]).float().half().to(torch.float64)
            leave = d[part] * tf[part, None]
            length = (leave - entry).norm(dim=1)
            steps = torch.floor(length / step).long() + 1
            a, b = ((p @ inv[:3, :3] + om - lo) * edge + 0.5 for p in (entry, leave))
            k = torch.arange(int(steps.max()), **f8)
            u = a[:, None] + k[:, None] * ((b - a) / (length / step)[:, None])[:, None]
            val = _lerp(brick, u)
            i = torch.floor((val * top / high).clamp(0, 1) * len(opaque)).long().clamp(max=len(opaque) - 1)
            if lit or two:
                grad = []
                for ax in range(3):
                    e = torch.zeros(3, **f8)
                    e[ax] = 1.0
                    grad.append((_lerp(brick, u - e) - _lerp(brick, u + e)) / 2)
                grad = torch.stack(grad, -1)
            if two:
                row = torch.floor((1 - grad.norm(dim=-1) * gscale).clamp(0, 1) * 256).long().clamp(max=255)
                s = table[row, i]
            else:
                s = table[i]
            rgb, alpha = s[..., :3], 1 - (1 - s[..., 3]) ** (1 / srm)
            if lit:
                nrm = grad @ mv[:3, :3]
                nrm = nrm / nrm.norm(dim=-1, keepdim=True).clamp(min=1e-300)
                pos = entry[:, None] + k[:, None] * ((leave - entry) / length[:, None] * step)[:, None]
                view = -pos / pos.norm(dim=-1, keepdim=True)
                mirror = view - nrm * (2 * (nrm * view).sum(-1, keepdim=True))
                spec = (mirror @ light).clamp(min=0) ** 8
                rgb = (amb + rgb * (nrm @ light).abs()[..., None] + spec[..., None]).clamp(0, 1)
            alpha = torch.where(k < steps[:, None], alpha, torch.zeros_like(alpha))
            through = torch.cumprod(1 - alpha, 1)
            before = torch.cat([torch.ones_like(through[:, :1]), through[:, :-1]], 1)
            ray = 1 - out[part, 3]
            stop = before <= 0.01
            if ert > 0:
                stop = stop | (ray[:, None] * before < ert)
            wgt = torch.where(stop & (k > 0), torch.zeros_like(alpha), alpha * before)
            seg = torch.cat([(wgt[..., None] * rgb).sum(1), wgt.sum(1, keepdim=True)], 1)
            out[part] += seg * ray[:, None]
    return out.reshape(H, W, 4)
