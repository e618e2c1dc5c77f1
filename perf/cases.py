"""The workloads that the library's speed is measured on, through its public entry points.

A case is one pass of a frame (or of a batch of frames) as a user's renderer calls it: single-frame
resolves with and without fused CAS over the frame sizes of the workloads module and ragged ones,
in both storages and both arithmetics; the reference's default parameter block; the upsampling
resolve; the resolve with the segmentation mask; the velocity producer; the edge-AA pass followed
by stand-alone sharpening; and a graph plan over the served resolution mix. Every input is made on
the GPU from the seed: layered moving discs and boxes with HDR luminance, their depth, velocity and
ids, and the previous frame as the history.

A single-frame pass reads the same history each time (it writes another buffer), so it can be
repeated; a batch pass advances its sessions, as a serving loop does.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "taa-star_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import taastar  # noqa: E402
from taastar import (ARITH_FP16, ARITH_FP32, FMT_RGBA16F, FMT_RGBA32F, VEL_RG16F, VEL_RG32F, VEL_RGBA16F,  # noqa: E402
                     VEL_RGBA32F, BatchItem, EdgeAaConsts, FrameImages, Reproject, SegmentationImages, SessionIO, Uniforms,
                     check, lib)

NEAR, FAR = 0.1, 100.0
SHARPNESS = 0.5
# the served resolution mix (40 / 35 / 15 / 10 %), dealt over any number of sessions
MIX = ((1280, 720), (1920, 1080), (1280, 720), (2560, 1440), (1920, 1080), (1280, 720), (1920, 1080), (3840, 2160),
       (1280, 720), (1920, 1080), (2560, 1440), (1280, 720))


# ---- the cases ----------------------------------------------------------------------------------

def listed():
    frame = dict(kind="frame", pitch=0, rgba_velocity=False)
    return [
        # the smallest call: a preview window, plain variance clip, no depth features, no sharpening
        dict(frame, name="frame_360p_fp32", w=640, h=360, half=False, arith="fp32", preset="plain", cas=False),
        # a game's frame at full precision, every feature of the production set, sharpened
        dict(frame, name="frame_1080p_fp32_cas", w=1920, h=1080, half=False, arith="fp32", preset="full", cas=True),
        # the throughput path at 4K: half storage and the FP16 arithmetic
        dict(frame, name="frame_4k_fp16_cas", w=3840, h=2160, half=True, arith="fp16", preset="full", cas=True),
        # a laptop window: odd height, rows padded to the allocator's pitch
        dict(frame, name="frame_1366x769_fp16_cas", w=1366, h=769, half=True, arith="fp16", preset="full", cas=True, pitch=1408),
        # a user who switches over with the reference's default parameter block and its RGBA16F
        # velocity image: first in the FP16 arithmetic, then in the exact one
        dict(frame, name="defaults_1440p_fp16_cas", w=2560, h=1440, half=True, arith="fp16", preset="defaults", cas=True,
             rgba_velocity=True),
        dict(frame, name="defaults_1080p_exact_cas", w=1920, h=1080, half=True, arith="fp32", preset="defaults", cas=True,
             rgba_velocity=True),
        # temporal upsampling: the usual 2x step to 4K, and an odd 1.5x one in the exact arithmetic
        dict(kind="upscale", name="upscale_1080p_to_4k_fp16", w=3840, h=2160, wl=1920, hl=1080, half=True, arith="fp16", cas=True),
        dict(kind="upscale", name="upscale_1281x721_exact", w=1921, h=1081, wl=1281, hl=721, half=False, arith="fp32", cas=True),
        # the resolve that also writes the ray tracer's segmentation mask
        dict(kind="mask", name="mask_1080p_fp32_cas", w=1920, h=1080, half=False, arith="fp32", cas=True),
        # a renderer without a velocity target: motion vectors from depth, with object ids
        dict(kind="velocity", name="velocity_4k_rgba16f", w=3840, h=2160, format="rgba16f", ids=True),
        # after a masked resolve: the edge-AA pass on category-1 texels, then sharpening on its own
        dict(kind="post", name="edge_aa_and_cas_1440p", w=2560, h=1440, half=True),
        # a server's round: a graph plan over twelve sessions of the served mix
        dict(kind="batch", name="batch_12_sessions_fp16", sessions=12, scale=1.0, half=True, arith="fp16", preset="full", cas=True),
    ]


def draw(rng):
    kind = rng.choice(("frame", "frame", "frame", "frame", "upscale", "mask", "velocity", "post", "batch"))
    w = int(round(math.exp(rng.uniform(math.log(320), math.log(3840)))))
    h = max(160, min(2160, int(round(w * rng.choice((9 / 16, 9 / 16, 10 / 16, 3 / 4, 9 / 21)))) + rng.randint(-3, 3)))
    half, arith = rng.choice(((True, "fp16"), (True, "fp16"), (True, "fp32"), (False, "fp32")))
    if kind == "frame":
        preset = rng.choice(("full", "full", "plain", "defaults"))
        return dict(kind=kind, w=w, h=h, half=half, arith=arith, preset=preset, cas=rng.random() < 0.75,
                    pitch=rng.choice((0, 0, (w + 63) // 64 * 64, w + rng.randint(1, 40))), rgba_velocity=preset == "defaults")
    if kind == "upscale":
        s = rng.choice((1.3, 1.5, 1.7, 2.0))
        w, h = max(w, 480), max(h, 270)
        return dict(kind=kind, w=w, h=h, wl=int(w / s), hl=int(h / s), half=half, arith=arith, cas=rng.random() < 0.75)
    if kind == "mask":
        w, h = min(w, 2560), min(h, 1600)
        return dict(kind=kind, w=w, h=h, half=half, arith=arith, cas=rng.random() < 0.75)
    if kind == "velocity":
        return dict(kind=kind, w=w, h=h, format=rng.choice(("rg16f", "rgba16f", "rg32f", "rgba32f")), ids=rng.random() < 0.6)
    if kind == "post":
        return dict(kind=kind, w=w, h=h, half=half)
    return dict(kind=kind, sessions=rng.randint(2, 12), scale=round(math.exp(rng.uniform(math.log(0.3), 0.0)), 3), half=True,
                arith="fp16", preset="full", cas=True)


def batch_sizes(case):
    return [(max(160, int(w * case["scale"])), max(90, int(h * case["scale"]))) for w, h in
            (MIX[i % len(MIX)] for i in range(case["sessions"]))]


# ---- scenes -------------------------------------------------------------------------------------

def _rng(seed):
    return np.random.default_rng(seed)


def _ndc(distance):
    """NDC depth (0 near, 1 far) of a view distance."""
    return FAR / (FAR - NEAR) - FAR * NEAR / (FAR - NEAR) / distance


def halton(i, b):
    f, r = 1.0, 0.0
    while i > 0:
        f /= b
        r += f * (i % b)
        i //= b
    return r


class Scene:
    """Layers of moving discs and boxes over a sloped background. frame(k) renders frame k at a
    sub-texel jitter; every layer is a grid of cells whose contents come from the seed."""

    LAYERS = ((240.0, 12.0, False), (90.0, 6.0, False), (30.0, 3.0, True))  # cell size, distance, moves on its own

    def __init__(self, w, h, seed, sigma=1.5):
        self.w, self.h, self.sigma = w, h, sigma
        r = _rng(seed)
        ang, mag = r.uniform(0, 2 * np.pi), r.uniform(1.0, 8.0) * w / 1920
        self.pan = np.array([np.cos(ang), 0.5 * np.sin(ang)]) * mag  # texels per frame
        self.own = self.pan + r.uniform(-6.0, 6.0, 2) * w / 1920
        t = r.random((4096, 10)).astype(np.float32)
        lum = np.exp(sigma * r.standard_normal(4096) - 1.2)
        t[:, 5:8] = (0.15 + 0.85 * t[:, 5:8]) * np.minimum(lum, 2000.0)[:, None]
        self.table = torch.from_numpy(t).cuda()
        self.off = int(r.integers(0, 4096))

    def frame(self, k, jitter=(0.0, 0.0)):
        """colour [h, w, 3] f32, depth [h, w] f32 (NDC), motion [h, w, 2] f32 (uv per frame), id [h, w] i32
        (0: static), cell [h, w] i32 (what a texel shows)."""
        w, h, dev = self.w, self.h, "cuda"
        x = (torch.arange(w, device=dev, dtype=torch.float32) + 0.5 + jitter[0])[None, :]
        y = (torch.arange(h, device=dev, dtype=torch.float32) + 0.5 + jitter[1])[:, None]
        sx, sy = x - float(self.pan[0]) * k, y - float(self.pan[1]) * k
        dist = (20.0 + 0.0005 * sy).expand(h, w)
        shade = 0.25 + 0.1 * torch.sin(sx * 0.21) * torch.sin(sy * 0.17)
        color = torch.stack((0.5 * shade, 0.6 * shade, 0.9 * shade), -1)
        cell = torch.zeros(h, w, dtype=torch.int32, device=dev)
        ident = torch.zeros(h, w, dtype=torch.int32, device=dev)
        motion = torch.tensor([self.pan[0] / w, self.pan[1] / h], dtype=torch.float32, device=dev).expand(h, w, 2)
        own = torch.tensor([self.own[0] / w, self.own[1] / h], dtype=torch.float32, device=dev)
        for n, (size, base, moves) in enumerate(self.LAYERS):
            v = self.own if moves else self.pan
            px, py = x - float(v[0]) * k, y - float(v[1]) * k
            cx, cy = torch.floor(px / size), torch.floor(py / size)
            fx, fy = px / size - cx, py / size - cy
            key = ((cx.int() * 7919 + cy.int() * 104729 + n * 1301 + self.off) & 4095).long()
            t = self.table[key]
            dx, dy = (fx - (0.4 + 0.2 * t[..., 1])).abs(), (fy - (0.4 + 0.2 * t[..., 2])).abs()
            rad = 0.15 + 0.22 * t[..., 3]
            inside = torch.where(t[..., 4] < 0.5, dx * dx + dy * dy < rad * rad, torch.maximum(dx, dy) < rad)
            d = base * (0.7 + 0.5 * t[..., 8])
            take = inside & (t[..., 0] < 0.6) & (d < dist)
            shade = 1.0 + 0.2 * torch.sin(px * 0.35) * torch.sin(py * 0.31)
            color = torch.where(take[..., None], t[..., 5:8] * shade[..., None], color)
            dist = torch.where(take, d, dist)
            cell = torch.where(take, (key + 1).int(), cell)
            if moves:
                ident = torch.where(take, (key % 7 + 1).int(), ident)
                motion = torch.where(take[..., None], own, motion)
        return color, _ndc(dist).float(), motion, ident, cell


def jitter_of(k, w, h):
    """Halton(2, 3) offsets of frame k, in texels and in NDC."""
    jx, jy = halton(k % 16 + 1, 2) - 0.5, halton(k % 16 + 1, 3) - 0.5
    return (jx, jy), (2.0 * jx / w, 2.0 * jy / h)


def _padded(a, pitch):
    """[h, w, ...] as an image of `pitch` texels a row."""
    if not pitch or pitch == a.shape[1]:
        return a.contiguous()
    out = torch.zeros((a.shape[0], pitch) + tuple(a.shape[2:]), dtype=a.dtype, device=a.device)
    out[:, : a.shape[1]] = a
    return out


def _rgba(color, alpha, half):
    c = torch.cat((color, torch.full_like(color[..., :1], alpha)), -1)
    return c.clamp(max=32768.0).half() if half else c


def frame_inputs(w, h, seed, half, rgba_velocity=False, wl=None, hl=None, sigma=1.5, k=1):
    """The images of frame k of a scene seen at w x h: current ones at wl x hl (the output size unless given)."""
    wl, hl = wl or w, hl or h
    low = Scene(wl, hl, seed, sigma)
    (jx, jy), ndc = jitter_of(k, wl, hl)
    color, depth, motion, ident, cell = low.frame(k, (jx, jy))
    _, pdepth, _, _, pcell = low.frame(k - 1, jitter_of(k - 1, wl, hl)[0])
    full = low
    if (wl, hl) != (w, h):  # the history of the same scene at the output size
        full = Scene(w, h, seed, sigma)
        full.LAYERS = tuple((s * w / wl, b, m) for s, b, m in Scene.LAYERS)
        full.pan, full.own = low.pan * w / wl, low.own * w / wl
    hist = full.frame(k - 1)[0]
    hist = 0.5 * hist + 0.25 * (torch.roll(hist, 1, 1) + torch.roll(hist, 1, 0))  # accumulated over jittered frames
    if rgba_velocity:
        vel = torch.cat((motion, torch.zeros_like(motion[..., :1]), ident[..., None].float()), -1)
    else:
        vel = motion
    vel = vel.half() if half else vel.float()
    return dict(color=_rgba(color, 1.0, half), depth=depth, prev_depth=pdepth, history=_rgba(hist, 0.0, half),
                velocity=vel.contiguous(), cell=cell, prev_cell=pcell, ident=ident, jitter=ndc, pan=low.pan)


# ---- parameters ---------------------------------------------------------------------------------

def params_of(preset):
    """The members of the Parameters block that differ from the reference's defaults."""
    if preset == "defaults":
        return {}
    p = dict(mVarianceClipping=1, mVarClipGamma=1.0, mColorClampingOrClipping=2, mInterpolationMode=2, mAlpha=0.1,
             mUseVelocityVectors=2, mVelocitySampleMode=0, mUseYCoCg=1)
    if preset != "plain":
        p.update(mVelocitySampleMode=2, mDepthCulling=1, mLumaWeightingLottes=1, mRejectOutside=1)
    if preset == "mask":
        p.update(mRayTraceAugment=1, mRayTraceHistoryCount=4)
    return p


def linear_threshold(preset):
    return 0.01 if preset in ("full", "mask") else 0.0


def matrices(w, h, pan):
    """Inverse view-projection of this frame and view-projection of the last (row-major float64): a camera that
    turned by what moves the background by `pan` texels at the frame's centre."""
    f, aspect = 1.0 / math.tan(math.radians(30.0)), w / h
    P = np.zeros((4, 4))
    P[0, 0], P[1, 1], P[2, 2], P[2, 3], P[3, 2] = f / aspect, f, FAR / (NEAR - FAR), -(FAR * NEAR) / (FAR - NEAR), -1.0
    yaw = math.atan(2.0 * pan[0] / w * aspect / f)
    pitch = math.atan(2.0 * pan[1] / h / f)
    cy, sy, cp, sp = math.cos(yaw), math.sin(yaw), math.cos(pitch), math.sin(pitch)
    Ry = np.array([[cy, 0, sy, 0], [0, 1, 0, 0], [-sy, 0, cy, 0], [0, 0, 0, 1.0]])
    Rx = np.array([[1, 0, 0, 0], [0, cp, -sp, 0], [0, sp, cp, 0], [0, 0, 0, 1.0]])
    return np.linalg.inv(P), P @ Ry @ Rx


def uniforms_of(preset, w, h, jitter, pan, upsampling=False, reset=False):
    U = Uniforms()
    p = taastar.default_params()
    for k, v in params_of(preset).items():
        setattr(p, k, v)
    U.param[0] = p
    U.param[1] = p
    Mi, Mh = matrices(w, h, pan)
    U.mInverseViewProjMatrix[:] = Mi.T.reshape(-1).astype(np.float32).tolist()
    U.mHistoryViewProjMatrix[:] = Mh.T.reshape(-1).astype(np.float32).tolist()
    U.mJitterNdc[0], U.mJitterNdc[1] = jitter
    U.mCamNearPlane, U.mCamFarPlane, U.pad1 = NEAR, FAR, linear_threshold(preset)
    U.mUpsampling, U.mResetHistory = int(upsampling), int(reset)
    return U


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


ARITH = {"fp32": ARITH_FP32, "fp16": ARITH_FP16}
VELOCITY = {"rg32f": (VEL_RG32F, 2, torch.float32), "rg16f": (VEL_RG16F, 2, torch.float16),
            "rgba32f": (VEL_RGBA32F, 4, torch.float32), "rgba16f": (VEL_RGBA16F, 4, torch.float16)}


def velocity_format(half, rgba):
    return VELOCITY[("rgba" if rgba else "rg") + ("16f" if half else "32f")][0]


def scene_of(case, seed):
    """The images of a frame, upscale or mask case."""
    sigma = 0.5 if case["kind"] == "mask" else 1.5
    return frame_inputs(case["w"], case["h"], seed, case["half"], case.get("rgba_velocity", False), case.get("wl"), case.get("hl"), sigma)


def mask_inputs(images, seed):
    """Material ids (bit 31: moving), the uv + normal-angle G-buffer and the last frame's mask."""
    def material(cell):
        m = cell.long() % 61 + 1
        return torch.where(m % 5 == 0, m | 0x80000000, m).to(torch.int64)

    def as_u32(m):
        return torch.where(m >= 2 ** 31, m - 2 ** 32, m).to(torch.int32).contiguous()

    cur, prev = material(images["cell"]), material(images["prev_cell"])
    h, w = cur.shape
    ids = (cur & 0x7fffffff).float()
    uvn = torch.empty(h, w, 4, dtype=torch.float32, device="cuda")
    uvn[..., 0] = ((torch.arange(w, device="cuda") + 0.5) / w)[None, :]
    uvn[..., 1] = ((torch.arange(h, device="cuda") + 0.5) / h)[:, None]
    uvn[..., 2] = torch.remainder(ids * 0.6180339887, 2 * math.pi)
    uvn[..., 3] = torch.remainder(ids * 0.3819660113, math.pi) - math.pi / 2
    marked = (images["cell"] != images["prev_cell"]) & (images["prev_cell"] % 3 == 0)
    prev_mask = torch.where(marked, torch.full_like(cur, (2 << 16) | 2), torch.zeros_like(cur)).to(torch.int32)
    return dict(material=as_u32(cur), prev_material=as_u32(prev), uv_normal=uvn, prev_mask=prev_mask)


def reproject_of(case, seed):
    """Camera matrices (row-major float64), jitters and seven object matrices of a velocity case."""
    r = _rng(seed + 17)
    w, h = case["w"], case["h"]
    Mi, Mp = matrices(w, h, r.uniform(-4.0, 4.0, 2) * w / 1920)
    jit = np.concatenate((r.uniform(-1, 1, 2) / (w, h), r.uniform(-1, 1, 2) / (w, h)))
    T = lambda x, y: np.array([[1, 0, x, 0], [0, 1, y, 0], [0, 0, 1, 0], [0, 0, 0, 1.0]])  # noqa: E731  jitter: NDC += j
    Mi, Mp = Mi @ np.linalg.inv(T(-jit[0], -jit[1])), T(-jit[2], -jit[3]) @ Mp
    objs = []
    for _ in range(7):
        a = r.uniform(-0.004, 0.004)
        o = np.array([[math.cos(a), 0, math.sin(a), 0], [0, 1, 0, 0], [-math.sin(a), 0, math.cos(a), 0], [0, 0, 0, 1.0]])
        o[:3, 3] = r.uniform(-0.01, 0.01, 3)
        objs.append(o)
    f32 = lambda m: m.astype(np.float32)  # noqa: E731
    return f32(Mi), f32(Mp), f32(jit), f32(np.stack(objs))


# ---- prepare ------------------------------------------------------------------------------------

class State:
    """What a pass needs, by name."""


def _frame_state(case, seed):
    w, h, half = case["w"], case["h"], case["half"]
    pitch = case.get("pitch") or w
    im = scene_of(case, seed)
    s = State()
    s.bufs = {k: _padded(im[k], pitch) for k in ("color", "depth", "prev_depth", "history", "velocity")} if "wl" not in case else \
        {k: im[k].contiguous() for k in ("color", "depth", "prev_depth", "history", "velocity")}
    dt = torch.float16 if half else torch.float32
    s.screen = torch.zeros(h, pitch, 4, dtype=dt, device="cuda")
    s.result = torch.zeros(h, pitch, 4, dtype=dt, device="cuda")
    img = FrameImages()
    img.color, img.depth, img.velocity = (s.bufs[k].data_ptr() for k in ("color", "depth", "velocity"))
    img.history, img.history_depth = s.bufs["history"].data_ptr(), s.bufs["prev_depth"].data_ptr()
    img.result_screen, img.result_history = s.screen.data_ptr(), s.result.data_ptr()
    img.width, img.height, img.pitch = w, h, pitch
    if "wl" in case:
        img.input_width, img.input_height, img.input_pitch = case["wl"], case["hl"], case["wl"]
    img.color_format = FMT_RGBA16F if half else FMT_RGBA32F
    img.velocity_format = velocity_format(half, case.get("rgba_velocity", False))
    preset = case.get("preset", "mask" if case["kind"] == "mask" else "full")
    U = uniforms_of(preset, w, h, im["jitter"], im["pan"], upsampling="wl" in case)
    k = taastar.cas_setup(SHARPNESS, w, h) if case["cas"] else None
    s.keep = (U, img, k)
    s.uniforms, s.images, s.cas = C.byref(U), C.byref(img), C.byref(k) if k is not None else None
    s.arith = ARITH[case["arith"]]
    if case["kind"] == "mask":
        m = mask_inputs(im, seed)
        s.mask = torch.zeros(h, pitch, dtype=torch.int32, device="cuda")
        seg = SegmentationImages()
        seg.material, seg.prev_material, seg.uv_normal = (m[k].data_ptr() for k in ("material", "prev_material", "uv_normal"))
        seg.prev_segmask, seg.segmask = m["prev_mask"].data_ptr(), s.mask.data_ptr()
        s.keep += (m, seg)
        s.seg = C.byref(seg)
    return s


class _View:
    """Device memory as torch.as_tensor takes it; the tensor keeps this object, and so the memory's owner."""


def _device_image(ptr, shape, dtype, owner):
    """A tensor over device memory of the library's, which `owner` keeps."""
    v = _View()
    v.owner = owner
    v.__cuda_array_interface__ = dict(shape=shape, typestr={torch.float16: "<f2", torch.float32: "<f4"}[dtype], data=(ptr, False),
                                      version=3, strides=None)
    return torch.as_tensor(v, device="cuda")


class Sessions:
    """A context, its sessions and a plan over them, given back when the last user of their memory is gone."""

    def __init__(self):
        self.ctx, self.plan, self.open = C.c_void_p(), C.c_void_p(), []
        check(lib().taa_ctx_create(0, 0, C.byref(self.ctx)))

    def add(self, w, h, fmt, vfmt):
        p = C.c_void_p()
        check(lib().taa_session_open(self.ctx, w, h, fmt, vfmt, C.byref(p)))
        self.open.append(p)
        return p

    def __del__(self):
        torch.cuda.synchronize()
        if self.plan:
            lib().taa_batch_plan_destroy(self.plan)
        for p in self.open:
            lib().taa_session_close(p)
        if self.ctx:
            lib().taa_ctx_destroy(self.ctx)


class Batch(State):
    """Sessions of one context and a graph plan over them; each holds frame 1 of its own scene, frame 0 resolved."""

    def __init__(self, case, seed):
        half, self.dtype = case["half"], torch.float16 if case["half"] else torch.float32
        self.sizes = batch_sizes(case)
        fmt, vfmt = (FMT_RGBA16F, VEL_RG16F) if half else (FMT_RGBA32F, VEL_RG32F)
        self.sessions, self.views, self.screens = Sessions(), {}, []
        n = len(self.sizes)
        self.items, self.uniforms, self.io = (BatchItem * n)(), (Uniforms * n)(), SessionIO()
        self.consts, ims = [], []
        for i, (w, h) in enumerate(self.sizes):
            p = self.sessions.add(w, h, fmt, vfmt)
            self.screens.append(torch.zeros(h, w, 4, dtype=self.dtype, device="cuda"))
            self.consts.append(taastar.cas_setup(SHARPNESS, w, h))
            im = batch_images(case, seed, i)
            ims.append(im)
            self.uniforms[i] = uniforms_of(case["preset"], w, h, im["jitter"], im["pan"])
            it = self.items[i]
            it.session, it.result_screen = p, self.screens[i].data_ptr()
            it.uniforms, it.cas = C.pointer(self.uniforms[i]), C.pointer(self.consts[i])
            self.fill(i, im["history"], im["prev_depth"], im["velocity"])
        check(lib().taa_batch_plan_create(self.sessions.ctx, n, self.items, ARITH[case["arith"]], C.byref(self.sessions.plan)))
        self.launch()
        for i, im in enumerate(ims):
            self.fill(i, im["color"], im["depth"], im["velocity"])

    def fill(self, i, color, depth, velocity):
        w, h = self.sizes[i]
        check(lib().taa_session_io(self.sessions.open[i], C.byref(self.io)))
        for p, a in ((self.io.color, color), (self.io.depth, depth), (self.io.velocity, velocity)):
            _device_image(p, tuple(a.shape), a.dtype, self.sessions).copy_(a)

    def launch(self):
        check(lib().taa_batch_plan_launch(self.sessions.plan, _stream()))

    def history(self, i):
        check(lib().taa_session_io(self.sessions.open[i], C.byref(self.io)))
        p = self.io.history
        if p not in self.views:
            w, h = self.sizes[i]
            self.views[p] = _device_image(p, (h, w, 4), self.dtype, self.sessions)
        return self.views[p]


def batch_images(case, seed, i):
    w, h = batch_sizes(case)[i]
    return frame_inputs(w, h, seed * 64 + i, case["half"])


def _velocity_state(case, seed):
    w, h = case["w"], case["h"]
    _, depth, _, ident, _ = Scene(w, h, seed).frame(1, jitter_of(1, w, h)[0])
    s = State()
    Mi, Mp, jit, objs = reproject_of(case, seed)
    fmt, ch, dt = VELOCITY[case["format"]]
    s.depth, s.ids = depth.contiguous(), ident.contiguous() if case["ids"] else None
    s.out = torch.zeros(h, w, ch, dtype=dt, device="cuda")
    s.objects = torch.from_numpy(np.ascontiguousarray(objs.transpose(0, 2, 1))).cuda()
    r = Reproject()
    r.inverse_view_proj[:] = Mi.T.reshape(-1).tolist()
    r.prev_view_proj[:] = Mp.T.reshape(-1).tolist()
    r.jitter_current_prev[:] = jit.tolist()
    if case["ids"]:
        r.object_prev_from_current, r.n_objects = s.objects.data_ptr(), objs.shape[0]
    s.keep, s.fmt, s.w, s.h = r, fmt, w, h
    s.args = (C.byref(r), C.c_void_p(s.depth.data_ptr()), None if s.ids is None else C.c_void_p(s.ids.data_ptr()),
              C.c_void_p(s.out.data_ptr()), fmt, w, h, w)
    return s


def post_inputs(case, seed):
    """A resolved screen and its mask: edges fall to the edge-AA pass where the history was off screen or rejected."""
    color, _, _, _, cell = Scene(case["w"], case["h"], seed, 0.5).frame(1)
    edge = torch.zeros_like(cell, dtype=torch.bool)
    edge[:, 1:] |= cell[:, 1:] != cell[:, :-1]
    edge[1:] |= cell[1:] != cell[:-1]
    edge[:, : case["w"] // 32] = True
    mask = torch.where(edge, 1, torch.where(cell % 13 == 1, 2 | (3 << 16), 0)).to(torch.int32)
    return _rgba(color, 1.0, case["half"]), mask.contiguous()


def _post_state(case, seed):
    w, h = case["w"], case["h"]
    s = State()
    s.src, s.mask = post_inputs(case, seed)
    s.smooth, s.out = torch.zeros_like(s.src), torch.zeros_like(s.src)
    e = EdgeAaConsts()
    check(lib().taa_edge_aa_defaults(w, h, C.byref(e)))
    k = taastar.cas_setup(SHARPNESS, w, h)
    s.keep = (e, k)
    fmt = FMT_RGBA16F if case["half"] else FMT_RGBA32F
    s.edge = (C.c_void_p(s.src.data_ptr()), C.c_void_p(s.mask.data_ptr()), C.c_void_p(s.smooth.data_ptr()), w, h, w, w, fmt, C.byref(e))
    s.cas = (C.c_void_p(s.smooth.data_ptr()), C.c_void_p(s.out.data_ptr()), w, h, w, fmt, C.byref(k))
    return s


def prepare(case, seed):
    s = {"frame": _frame_state, "upscale": _frame_state, "mask": _frame_state, "velocity": _velocity_state, "post": _post_state,
         "batch": Batch}[case["kind"]](case, seed)
    s.kind = case["kind"]
    return s


# ---- run ----------------------------------------------------------------------------------------

def run(s):
    if s.kind in ("frame", "upscale"):
        check(lib().taa_resolve_frame(s.uniforms, s.images, s.cas, s.arith, _stream()))
        return {"history": s.result, "screen": s.screen}
    if s.kind == "mask":
        check(lib().taa_resolve_frame_segmented(s.uniforms, s.images, s.seg, s.cas, s.arith, _stream()))
        return {"history": s.result, "screen": s.screen, "mask": s.mask}
    if s.kind == "velocity":
        check(lib().taa_velocity_from_depth(*s.args, _stream()))
        return {"velocity": s.out}
    if s.kind == "post":
        st = _stream()
        check(lib().taa_edge_aa_apply(*s.edge, st))
        check(lib().taa_cas_apply(*s.cas, st))
        return {"smooth": s.smooth, "screen": s.out}
    s.launch()
    return {"%02d" % i: {"history": s.history(i), "screen": s.screens[i]} for i in range(len(s.sizes))}


def work(case):
    """Bytes: each input read once, each output written once. flops: the arithmetic of one texel as
    the reference's shader states it (box, history filter, rejection, blend, sharpening), about."""
    if case["kind"] == "batch":
        px = sum(w * h for w, h in batch_sizes(case))
        return {"bytes": px * 44.0, "flops": px * 330.0}
    px = case["w"] * case["h"]
    if case["kind"] == "velocity":
        vb = {"rg32f": 8, "rg16f": 4, "rgba32f": 16, "rgba16f": 8}[case["format"]]
        return {"bytes": px * (4.0 + 4 * case["ids"] + vb), "flops": px * 70.0}
    cb = 8 if case["half"] else 16
    if case["kind"] == "post":
        return {"bytes": px * (4.0 * cb + 4), "flops": px * 40.0}
    low = case["wl"] * case["hl"] if "wl" in case else px
    vb = cb // 2 * (2 if case.get("rgba_velocity") else 1)
    preset = case.get("preset", "full")
    b = low * (cb + vb) + px * 3.0 * cb  # colour and velocity; history in and out, screen
    b += {"plain": 0, "defaults": 4}.get(preset, 8) * low  # depth, previous depth
    if case["kind"] == "mask":
        b += px * (4 + 4 + 16 + 4 + 4)
    return {"bytes": float(b), "flops": px * (280.0 + 50.0 * case["cas"])}


# ---- 64-bit values ------------------------------------------------------------------------------

def _f32_bits(x):
    return x.float().contiguous().view(torch.int32)


def _from_bits(b):
    return b.view(torch.float32).double()


def _clamped(img, dx, dy):
    """img shifted so that texel (x, y) holds texel (x + dx, y + dy), clamped to the edge."""
    h, w = img.shape[:2]
    iy = (torch.arange(h, device=img.device) + dy).clamp(0, h - 1)
    ix = (torch.arange(w, device=img.device) + dx).clamp(0, w - 1)
    return img[iy][:, ix]


def _cas64(c):
    """Contrast-adaptive sharpening of rgb [h, w, 3]; its reciprocals and square root are the filter's own integer steps."""
    b, d, f, e2 = _clamped(c, 0, -1), _clamped(c, -1, 0), _clamped(c, 1, 0), _clamped(c, 0, 1)
    g = torch.stack((b[..., 1], d[..., 1], c[..., 1], f[..., 1], e2[..., 1]))
    mx, mn = g.amax(0), g.amin(0)
    amp = (torch.minimum(mn, 1.0 - mx) * _from_bits(0x7ef07ebb - _f32_bits(mx))).clamp(0.0, 1.0)
    amp = _from_bits((_f32_bits(amp) >> 1) + 0x1fbc4639)
    peak = -1.0 / (8.0 * (1.0 - SHARPNESS) + 5.0 * SHARPNESS)
    w = amp * peak
    q = 1.0 + 4.0 * w
    r = _from_bits(0x7ef19fff - _f32_bits(q))
    rw = r * (2.0 - r * q)
    o = ((b + d + f + e2) * w[..., None] + c) * rw[..., None]
    return torch.cat((o.clamp(0.0, 1.0), torch.ones_like(o[..., :1])), -1)


def _ycocg(c):
    r, g, b = c.unbind(-1)
    return torch.stack((0.25 * r + 0.5 * g + 0.25 * b, 0.5 * r - 0.5 * b, -0.25 * r + 0.5 * g - 0.25 * b), -1)


def _rgb(c):
    y, co, cg = c.unbind(-1)
    return torch.stack((y - cg + co, y + cg, y - cg - co), -1)


def _linear(d):
    return NEAR * FAR / (FAR + d * (NEAR - FAR))


def _gather(img, ix, iy):
    h, w = img.shape[:2]
    flat = img.reshape(h * w, -1)
    return flat[(iy.clamp(0, h - 1) * w + ix.clamp(0, w - 1)).reshape(-1)].reshape(ix.shape + (flat.shape[1],))


def _bilinear(img, u, v):
    """img [h, w, c] at (u, v), clamped to the edge, exact weights."""
    h, w = img.shape[:2]
    px, py = u * w - 0.5, v * h - 0.5
    fx, fy = torch.floor(px), torch.floor(py)
    tx, ty = (px - fx)[..., None], (py - fy)[..., None]
    ix, iy = fx.long(), fy.long()
    top = _gather(img, ix, iy) * (1 - tx) + _gather(img, ix + 1, iy) * tx
    return top * (1 - ty) + (_gather(img, ix, iy + 1) * (1 - tx) + _gather(img, ix + 1, iy + 1) * tx) * ty


def _catmull_rom(img, hu, hv):
    h, w = img.shape[:2]
    px, py = hu * w - 0.5, hv * h - 0.5
    bx, by = torch.floor(px), torch.floor(py)

    def weights(f):
        return (-0.5 * f ** 3 + f ** 2 - 0.5 * f, 1.5 * f ** 3 - 2.5 * f ** 2 + 1.0, -1.5 * f ** 3 + 2.0 * f ** 2 + 0.5 * f,
                0.5 * f ** 3 - 0.5 * f ** 2)
    wx, wy = weights(px - bx), weights(py - by)
    ix, iy, acc = bx.long(), by.long(), 0.0
    for j in range(4):
        for i in range(4):
            acc = acc + _gather(img, ix + (i - 1), iy + (j - 1)) * (wx[i] * wy[j])[..., None]
    return acc


def _sample_axis(l, h, jitter):
    """For each output column the input column of the jittered sample that falls into it, or -1 (taa.comp:222-257). Which
    texel it is comes from single-precision positions, so it is found in those."""
    f = np.float32
    tc, sc, tj = np.arange(h, dtype=np.float32), f(h) / f(l), f(jitter) * f(0.5) * f(l) * f(-1.0)
    pick, found = np.zeros(h, np.float32), np.zeros(h, bool)
    for o in (f(0.0), f(0.999999)):
        s = np.floor(f(l) * (tc + o) / f(h)) + f(0.5) + tj
        hit = (s * sc).astype(np.int32) == tc.astype(np.int32)
        pick, found = np.where(hit, s, pick).astype(np.float32), found | hit
    return np.where(found & (pick >= 0), np.clip(np.floor(pick), 0, l - 1), -1).astype(np.int64)


def _mask64(P, color, depth, m, hu, hv):
    """The segmentation mask's value per texel (int64)."""
    h, w = depth.shape
    mat = m["material"].long() & 0xffffffff
    count = P["mRayTraceHistoryCount"] << 16

    def sobel(t):
        a = {(x, y): _clamped(t, x, y) for x in (-1, 0, 1) for y in (-1, 0, 1)}
        gx = (a[-1, -1] - a[-1, 1]) + 2 * (a[0, -1] - a[0, 1]) + (a[1, -1] - a[1, 1])
        gy = (a[-1, -1] - a[1, -1]) + 2 * (a[-1, 0] - a[1, 0]) + (a[-1, 1] - a[1, 1])
        return torch.sqrt(gx * gx + gy * gy)
    q = m["uv_normal"].double()
    n = torch.stack((torch.cos(q[..., 2]) * torch.cos(q[..., 3]), torch.sin(q[..., 2]) * torch.cos(q[..., 3]), torch.sin(q[..., 3])), -1)
    cross = ((-1, 0), (1, 0), (0, -1), (0, 1))
    dots = torch.stack([(n * _clamped(n, x, y)).sum(-1) for x, y in cross]).amin(0).clamp(min=0.0)
    mid = torch.stack([mat != _clamped(mat, x, y) for x, y in cross]).any(0)
    total = (1.0 - dots) * P["mRayTraceAugment_WNrm"] + sobel(_linear(depth)) * P["mRayTraceAugment_WDpt"] + \
        mid.double() * P["mRayTraceAugment_WMId"] + sobel(_ycocg(color)[..., 0]) * P["mRayTraceAugment_WLum"]
    old = (m["prev_mask"].long() & 0xffff0000) >> 16
    v = torch.where(old > 0, 2 | ((old - 1) << 16), torch.zeros_like(old))
    v = torch.where(total >= P["mRayTraceAugment_Thresh"], torch.full_like(v, 2 | count), v)
    tx, ty = torch.trunc(hu * w).long(), torch.trunc(hv * h).long()
    prev = _gather((m["prev_material"].long() & 0xffffffff)[..., None], tx, ty)[..., 0]
    inside = (tx >= 0) & (ty >= 0) & (tx < w) & (ty < h)
    v = torch.where(inside & (prev != mat) & (prev >= 2 ** 31), torch.full_like(v, 2 | count), v)
    return torch.where((hu < 0) | (hv < 0) | (hu >= 1) | (hv >= 1), torch.ones_like(v), v)


def _resolve64(preset, im, w, h, cas, upsampling=False, mask=None):
    """history and screen [h, w, 4] of one frame."""
    P = {k: getattr(taastar.default_params(), k) for k, _ in taastar.Params._fields_}
    P.update(params_of(preset))
    color, history = im["color"][..., :3].double(), im["history"][..., :3].double()
    depth, pdepth, vel = im["depth"].double(), im["prev_depth"].double(), im["velocity"].double()
    hl, wl = depth.shape
    to = _ycocg if P["mUseYCoCg"] else (lambda c: c)
    cur = to(color)
    u = ((torch.arange(w, device="cuda", dtype=torch.float64) + 0.5) / w)[None, :].expand(h, w)
    v = ((torch.arange(h, device="cuda", dtype=torch.float64) + 0.5) / h)[:, None].expand(h, w)
    offsets = [(x, y) for y in (-1, 0, 1) for x in (-1, 0, 1)]
    taps = [_clamped(cur, x, y) for x, y in offsets]
    if P["mVarianceClipping"]:
        mean = sum(taps) / 9.0
        sigma = torch.sqrt((sum(t * t for t in taps) / 9.0 - mean * mean).clamp(min=0.0)) * P["mVarClipGamma"]
        lo, hi = mean - sigma, mean + sigma
    else:
        lo, hi = torch.stack(taps).amin(0), torch.stack(taps).amax(0)
    del taps
    beta = torch.ones(h, w, dtype=torch.float64, device="cuda")
    if upsampling:
        xl, yl = torch.trunc(u * wl).long(), torch.trunc(v * hl).long()
        lo, hi = _gather(lo, xl, yl), _gather(hi, xl, yl)
        d = _gather(depth[..., None], xl, yl)[..., 0]
        cx = torch.from_numpy(_sample_axis(wl, w, im["jitter"][0])).cuda()[None, :].expand(h, w)
        cy = torch.from_numpy(_sample_axis(hl, h, im["jitter"][1])).cuda()[:, None].expand(h, w)
        got = (cx >= 0) & (cy >= 0)
        beta = got.double()
        cur = _gather(cur, cx, cy) * beta[..., None]
    else:
        d = depth
    if P["mVelocitySampleMode"] == 2:
        best, vs = None, None
        for x, y in offsets:
            dk = _bilinear(depth[..., None], u + x / wl, v + y / hl)[..., 0] if upsampling else _clamped(depth, x, y)
            vk = _bilinear(vel, u + x / wl, v + y / hl) if upsampling else _clamped(vel, x, y)
            if best is None:
                best, vs = dk, vk
            else:
                take = dk < best
                best, vs = torch.where(take, dk, best), torch.where(take[..., None], vk, vs)
    else:
        vs = vel
    hu, hv = u - vs[..., 0], v - vs[..., 1]
    expected = d - (vs[..., 2] if vs.shape[-1] == 4 else 0.0)
    if P["mUseVelocityVectors"] == 1:  # movers by their velocity, the rest through the matrices
        Mi, Mh = (torch.from_numpy(m.astype(np.float32).astype(np.float64)).cuda() for m in matrices(w, h, im["pan"]))
        clip = torch.stack((u * 2 - 1, v * 2 - 1, d, torch.ones_like(d)), -1) @ Mi.T @ Mh.T
        moves = vel[..., 3] >= 0.5
        hu = torch.where(moves, hu, clip[..., 0] / clip[..., 3] * 0.5 + 0.5)
        hv = torch.where(moves, hv, clip[..., 1] / clip[..., 3] * 0.5 + 0.5)
        expected = torch.where(moves, expected, clip[..., 2] / clip[..., 3])
    old = to(_catmull_rom(history, hu, hv) if P["mInterpolationMode"] == 2 else _bilinear(history, hu, hv))
    rejected = torch.zeros(h, w, dtype=torch.bool, device="cuda")
    seg = None
    if mask is not None:
        seg = _mask64(P, color, depth, mask, hu, hv)
        rejected |= (seg & 3) != 0
    if P["mRejectOutside"]:
        rejected |= (hu < 0) | (hv < 0) | (hu >= 1) | (hv >= 1)
    if P["mDepthCulling"]:
        seen = _gather(pdepth[..., None], torch.trunc(hu * wl).long(), torch.trunc(hv * hl).long())[..., 0]
        rejected |= (_linear(seen) - _linear(expected)).abs() > linear_threshold(preset)
    if P["mColorClampingOrClipping"] == 1:
        old = torch.minimum(torch.maximum(old, lo), hi)
    else:
        c, e = 0.5 * (hi + lo), 0.5 * (hi - lo) + 1e-7
        ma = ((old - c) / e).abs().amax(-1, keepdim=True)
        old = torch.where(ma > 1.0, c + (old - c) / ma, old)
    alpha = torch.full((h, w), float(P["mAlpha"]), dtype=torch.float64, device="cuda")
    if P["mLumaWeightingLottes"]:
        luma = (lambda c: c[..., 0]) if P["mUseYCoCg"] else (lambda c: _ycocg(c)[..., 0])
        lc, lh = luma(cur), luma(old)
        k = 1.0 - (lc - lh).abs() / torch.maximum(lc, lh).clamp(min=0.2)
        alpha = P["mMaxAlpha"] + (P["mMinAlpha"] - P["mMaxAlpha"]) * k * k
    ab = torch.where(rejected, torch.full_like(alpha, float(P["mRejectionAlpha"])), alpha * beta)[..., None]
    out = old + (cur - old) * ab
    out = _rgb(out) if P["mUseYCoCg"] else out
    screen = _cas64(out) if cas else torch.cat((out, torch.ones_like(out[..., :1])), -1)
    return torch.cat((out, torch.zeros_like(out[..., :1])), -1), screen


def _velocity64(case, seed):
    w, h = case["w"], case["h"]
    _, depth, _, ident, _ = Scene(w, h, seed).frame(1, jitter_of(1, w, h)[0])
    Mi, Mp, jit, objs = (torch.from_numpy(a.astype(np.float64)).cuda() for a in reproject_of(case, seed))
    d = depth.double()
    x = (((torch.arange(w, device="cuda", dtype=torch.float64) + 0.5) / w) * 2 - 1)[None, :].expand(h, w)
    y = (((torch.arange(h, device="cuda", dtype=torch.float64) + 0.5) / h) * 2 - 1)[:, None].expand(h, w)
    world = torch.stack((x, y, d, torch.ones_like(d)), -1) @ Mi.T
    if case["ids"]:
        for k in range(objs.shape[0]):
            world = torch.where((ident == k + 1)[..., None], world @ objs[k].T, world)
    p = world @ Mp.T
    p = p[..., :3] / p[..., 3:]
    out = [((x - jit[0]) - (p[..., 0] - jit[2])) * 0.5, ((y - jit[1]) - (p[..., 1] - jit[3])) * 0.5]
    if case["format"].startswith("rgba"):
        out += [d - p[..., 2], ident.double() if case["ids"] else torch.zeros_like(d)]
    return torch.stack(out, -1)


def _post64(case, seed):
    src, mask = post_inputs(case, seed)
    c = src[..., :3].double()
    luma = c @ torch.tensor([0.299, 0.587, 0.114], dtype=torch.float64, device="cuda")
    l = {(x, y): _clamped(luma, x, y) for x in (-1, 0, 1) for y in (-1, 0, 1)}
    cross = torch.stack((luma, l[0, -1], l[0, 1], l[-1, 0], l[1, 0]))
    mn, mx = cross.amin(0), cross.amax(0)
    span = mx - mn
    gx = l[1, -1] + 2 * l[1, 0] + l[1, 1] - l[-1, -1] - 2 * l[-1, 0] - l[-1, 1]
    gy = l[-1, 1] + 2 * l[0, 1] + l[1, 1] - l[-1, -1] - 2 * l[0, -1] - l[1, -1]
    up = (l[0, -1] - luma).abs() >= (l[0, 1] - luma).abs()
    left = (l[-1, 0] - luma).abs() >= (l[1, 0] - luma).abs()
    vert = torch.where(up[..., None], _clamped(c, 0, -1), _clamped(c, 0, 1))
    hori = torch.where(left[..., None], _clamped(c, -1, 0), _clamped(c, 1, 0))
    other = torch.where((gy.abs() >= gx.abs())[..., None], vert, hori)
    avg = ((l[0, -1] + l[0, 1] + l[-1, 0] + l[1, 0]) * 2 + l[-1, -1] + l[1, -1] + l[-1, 1] + l[1, 1]) / 12.0
    hit = ((mask & 3) == 1) & (span >= torch.maximum(torch.full_like(mx, 0.0833), mx * 0.116)) & (span > 0)
    blend = torch.where(hit, 0.375 * ((avg - luma).abs() / span.clamp(min=1e-30)).clamp(0.0, 1.0), torch.zeros_like(span))[..., None]
    out = c * (1 - blend) + other * blend
    return torch.cat((out, luma[..., None]), -1), _cas64(out)


def exact(case, seed):
    if case["kind"] == "velocity":
        return {"velocity": _velocity64(case, seed)}
    if case["kind"] == "post":
        smooth, screen = _post64(case, seed)
        return {"smooth": smooth, "screen": screen}
    if case["kind"] == "batch":
        got = {}
        for i, (w, h) in enumerate(batch_sizes(case)):
            hist, screen = _resolve64(case["preset"], batch_images(case, seed, i), w, h, case["cas"])
            got["%02d" % i] = {"history": hist, "screen": screen}
        return got
    im = scene_of(case, seed)
    preset = case.get("preset", "mask" if case["kind"] == "mask" else "full")
    m = mask_inputs(im, seed) if case["kind"] == "mask" else None
    hist, screen = _resolve64(preset, im, case["w"], case["h"], case["cas"], "wl" in case, m)
    hist, screen = _padded(hist, case.get("pitch")), _padded(screen, case.get("pitch"))
    return {"history": hist, "screen": screen, "mask": None} if m else {"history": hist, "screen": screen}
