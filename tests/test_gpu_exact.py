"""The exact kernel of the production feature set against the general form (which a bound debug image selects): the same
bits, single frames and batches, on both sides of the line that selects it."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from gpu_helpers import assert_same_bits  # noqa: E402
from test_gpu_upscale import inputs, test_batches_equal_sessions_alone as batches  # noqa: E402
from taastar import (ARITH_FP16, ARITH_FP32, FMT_RGBA16F, FMT_RGBA32F, RTFLAG, VEL_RG16F, VEL_RG32F, VEL_RGBA16F, FrameImages,  # noqa: E402
                     SegmentationImages, check, default_params, lib)
from taastar.workloads import cas_for, uniforms_for, workload  # noqa: E402


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def both_forms(w, U, W, H, pitch, images, fmt, K, arith=ARITH_FP32, seg=None):
    """Screen and history of the frame without and with a debug image; seg: the mask's images, its output too."""
    color, depth, vel, hist, prev = images
    out = []
    for general in (False, True):
        screen, new = torch.zeros_like(hist), torch.zeros_like(hist)
        debug = torch.zeros(H, pitch, 4, dtype=torch.float16, device="cuda")
        img = FrameImages()
        img.color, img.depth, img.velocity = color.data_ptr(), depth.data_ptr(), vel.data_ptr()
        img.history, img.history_depth = hist.data_ptr(), prev.data_ptr()
        img.result_history, img.result_screen = new.data_ptr(), screen.data_ptr()
        img.debug = debug.data_ptr() if general else None
        img.width, img.height, img.pitch = W, H, pitch
        img.color_format, img.velocity_format = fmt, w["vel"]
        mask = torch.full((H, pitch), 7, dtype=torch.int32, device="cuda")
        if seg is None:
            check(lib().taa_resolve_frame(C.byref(U), C.byref(img), C.byref(K) if K else None, arith, None))
        else:
            g = SegmentationImages()
            g.material, g.prev_material, g.uv_normal, g.prev_segmask = [t.data_ptr() for t in seg]
            g.segmask, g.pitch, g.input_pitch = mask.data_ptr(), pitch, seg[0].shape[1]
            check(lib().taa_resolve_frame_segmented(C.byref(U), C.byref(img), C.byref(g), C.byref(K) if K else None, arith, None))
        torch.cuda.synchronize()
        out.append((screen, new, mask))
    assert torch.equal(out[0][2], out[1][2]), "mask"
    assert_same_bits(out[0][0], out[1][0], "screen")
    assert_same_bits(out[0][1], out[1][1], "history")


# regions are 30 x 14 (CAS) or 32 x 16 texels, 900 to 1500 of them select the kernel; the second size is a texel beyond
# whole regions, the last columns and rows of the third are one texel of a region; motion within the window and beyond it
@pytest.mark.parametrize("W,H,motion,odd", [(960, 540, 0, False), (1441, 897, 6, True), (961, 1121, 6, True), (1280, 720, 60, False),
                                            (3, 24001, 4, False), (24001, 3, 4, True), (333, 111, 6, True)])
@pytest.mark.parametrize("fmt", [FMT_RGBA16F, FMT_RGBA32F])
def test_equals_the_general_form(W, H, motion, odd, fmt):
    for k, (cas, pad, reset, split) in enumerate([(True, 0, 0, 0), (False, 3, 0, 0), (True, 5, 0, W // 3), (True, 0, 1, 0)]):
        print(f"case {W}x{H} fmt {fmt} cas {cas} pad {pad} reset {reset} split {split}", flush=True)
        w = workload("c2", fmt=fmt, vel=VEL_RG16F if fmt == FMT_RGBA16F else VEL_RG32F)
        U = uniforms_for(w, 1, (0.3 / W, -0.4 / H))
        U.mResetHistory, U.splitScreen, U.splitX = reset, int(split > 0), split
        both_forms(w, U, W, H, W + pad, inputs(W, H, W, H, W + pad, W + pad, fmt, motion, odd, 71 + k), fmt, cas_for(w, W, H) if cas else None)


# one row a thread below 800 regions (the first two sizes), two rows above; still texels are reprojected through the matrices
@pytest.mark.parametrize("W,H,odd", [(95, 61, True), (3, 2, False), (1281, 721, True), (31, 24001, False)])
def test_default_block_equals_the_general_form(W, H, odd):
    for k, (cas, pad, reset, split) in enumerate([(True, 0, 0, 0), (False, 3, 0, 0), (True, 5, 0, W // 3), (True, 0, 1, 0)]):
        print(f"case defaults {W}x{H} cas {cas} pad {pad} reset {reset} split {split}", flush=True)
        w = workload("c2", fmt=FMT_RGBA16F, vel=VEL_RGBA16F)
        U = uniforms_for(w, 1, (0.3 / W, -0.4 / H), params=default_params())
        U.mHistoryViewProjMatrix[12], U.mHistoryViewProjMatrix[5], U.mHistoryViewProjMatrix[11] = 0.01, 0.98, 0.02
        U.mResetHistory, U.splitScreen, U.splitX = reset, int(split > 0), split
        color, depth, vel, hist, prev = inputs(W, H, W, H, W + pad, W + pad, FMT_RGBA16F, 5, odd, 91 + k)
        moving = (torch.arange(W + pad, device="cuda") // 7 % 3 > 0).to(vel.dtype).expand(H, -1)
        vel4 = torch.stack([vel[..., 0], vel[..., 1], torch.full_like(moving, 0.001), moving], -1).contiguous()
        both_forms(w, U, W, H, W + pad, (color, depth, vel4, hist, prev), FMT_RGBA16F, cas_for(w, W, H) if cas else None)


def plain_params():
    p = workload("c2")["params"]()
    p.mVelocitySampleMode = p.mDepthCulling = p.mLumaWeightingLottes = p.mRejectOutside = 0
    return p


# without CAS one row a thread below 800 regions (the first three sizes), two rows above and with CAS
@pytest.mark.parametrize("W,H,motion,odd", [(1, 1, 0, False), (33, 17, 6, True), (95, 61, 40, False), (1281, 721, 6, True), (31, 24001, 4, False)])
@pytest.mark.parametrize("fmt", [FMT_RGBA16F, FMT_RGBA32F])
def test_plain_form_equals_the_general_form(W, H, motion, odd, fmt):
    for k, (cas, pad, reset, split) in enumerate([(True, 0, 0, 0), (False, 3, 0, 0), (True, 5, 0, W // 3), (False, 0, 1, 0)]):
        print(f"case plain {W}x{H} fmt {fmt} cas {cas} pad {pad} reset {reset} split {split}", flush=True)
        w = workload("c2", fmt=fmt, vel=VEL_RG16F if fmt == FMT_RGBA16F else VEL_RG32F)
        U = uniforms_for(w, 1, (0.3 / W, -0.4 / H), params=plain_params())
        U.mResetHistory, U.splitScreen, U.splitX = reset, int(split > 0), split
        both_forms(w, U, W, H, W + pad, inputs(W, H, W, H, W + pad, W + pad, fmt, motion, odd, 171 + k), fmt, cas_for(w, W, H) if cas else None)


@pytest.mark.parametrize("fmt", [FMT_RGBA16F, FMT_RGBA32F])
def test_plain_batches(fmt, monkeypatch):
    import test_gpu_upscale as t
    monkeypatch.setattr(t, "uniforms_for", lambda w, f, j: uniforms_for(w, f, j, params=plain_params()))
    batches([((480, 270), (480, 270)), ((33, 65), (33, 65))], fmt, ARITH_FP32)


@pytest.mark.parametrize("specs", [[((480, 270), (480, 270)), ((640, 361), (640, 361)), ((33, 65), (33, 65))],
                                   [((160, 90), (160, 90)), ((95, 61), (95, 61))]])
@pytest.mark.parametrize("fmt", [FMT_RGBA16F, FMT_RGBA32F])
def test_batches(specs, fmt):
    batches(specs, fmt, ARITH_FP32)


@pytest.mark.parametrize("specs", [[((480, 270), (480, 270)), ((33, 65), (33, 65))], [((960, 541), (960, 541)), ((640, 361), (640, 361))]])
def test_default_block_batches(specs, monkeypatch):
    import test_gpu_upscale as t
    rgba = lambda *a, **k: (lambda i: (i[0], i[1], torch.cat([i[2], i[2].abs() * 50], -1).contiguous(), i[3], i[4]))(inputs(*a, **k))
    monkeypatch.setattr(t, "inputs", rgba)
    monkeypatch.setattr(t, "VEL_RG16F", VEL_RGBA16F)
    monkeypatch.setattr(t, "uniforms_for", lambda w, f, j: uniforms_for(w, f, j, params=default_params()))
    batches(specs, FMT_RGBA16F, ARITH_FP32)


F = RTFLAG
FLAGS = [F["OUT"] | F["DIS"] | F["NRM"] | F["DPT"] | F["MID"] | F["LUM"] | F["CNT"], F["DPT"] | F["LUM"], F["OUT"] | F["DIS"] | F["MID"],
         F["NRM"] | F["CNT"] | F["FXD"], F["ALL"], F["ALL"] | F["FXD"] | F["OUT"] | F["DIS"], 0]


# 700 regions select the kernel: one region wide and high, inner tiles beyond the 100-texel border of FXD, and below the line
@pytest.mark.parametrize("W,H,odd", [(5, 12001, True), (22801, 7, False), (1021, 701, True), (61, 29, False)])
@pytest.mark.parametrize("fmt,arith", [(FMT_RGBA16F, ARITH_FP16), (FMT_RGBA16F, ARITH_FP32), (FMT_RGBA32F, ARITH_FP16), (FMT_RGBA32F, ARITH_FP32)])
def test_mask_equals_the_general_form(W, H, odd, fmt, arith):
    for k, flags in enumerate(FLAGS):
        cas, pad, split = k % 3 != 1, k % 2 * 3, W // 3 if k == 3 else 0
        print(f"case mask {W}x{H} fmt {fmt} arith {arith} flags {flags:#x} cas {cas} pad {pad} split {split}", flush=True)
        w = workload("c2", fmt=fmt, vel=VEL_RG16F if fmt == FMT_RGBA16F else VEL_RG32F)
        p = w["params"]()
        p.mRayTraceAugment, p.mRayTraceAugmentFlags, p.mRayTraceHistoryCount = 1, flags, 4
        U = uniforms_for(w, 1, (0.3 / W, -0.4 / H), params=p)
        U.splitScreen, U.splitX = int(split > 0), split
        pitch, spl = W + pad, W + 2 * pad
        images = inputs(W, H, W, H, pitch, pitch, fmt, 4, odd, 131 + k)
        g = torch.Generator(device="cuda").manual_seed(k)
        cells = torch.randint(0, 5, ((H + 4) // 5, (spl + 6) // 7), generator=g, device="cuda").repeat_interleave(5, 0).repeat_interleave(7, 1)[:H, :spl]
        moved = torch.rand(H, spl, generator=g, device="cuda") < 0.05
        material = cells.to(torch.int32).contiguous()
        prev = torch.where(moved, cells + 1, cells).to(torch.int32) | torch.where(cells % 2 == 0, -2**31, 0).to(torch.int32)
        normals = (cells[..., None].float() + 0.2 * torch.rand(H, spl, 4, generator=g, device="cuda")).contiguous()
        old = torch.where(torch.rand(H, pitch, generator=g, device="cuda") < 0.1, (3 << 16) | 2, 0).to(torch.int32)
        both_forms(w, U, W, H, pitch, images, fmt, cas_for(w, W, H) if cas else None, arith, (material, prev.contiguous(), normals, old))


@pytest.mark.parametrize("lo,W,H", [((960, 541), 960, 541), ((480, 270), 961, 541)])
@pytest.mark.parametrize("fmt,arith", [(FMT_RGBA16F, ARITH_FP16), (FMT_RGBA16F, ARITH_FP32), (FMT_RGBA32F, ARITH_FP32)])
def test_images_at_any_element(lo, W, H, fmt, arith):
    """Images that begin one element into their allocation give the results of aligned ones."""
    print(f"case alignment {lo} -> {W}x{H} fmt {fmt} arith {arith}", flush=True)
    w = workload("c2", fmt=fmt, vel=VEL_RG16F if fmt == FMT_RGBA16F else VEL_RG32F)
    U = uniforms_for(w, 1, (0.2 / W, 0.1 / H))
    U.mUpsampling = int(lo != (W, H))
    K = cas_for(w, W, H)
    images = inputs(*lo, W, H, lo[0], W, fmt, 4, False, 7)

    def moved(t, by):
        s = torch.zeros(t.numel() + by, dtype=t.dtype, device="cuda")
        s[by:] = t.reshape(-1)
        return s

    out = []
    for by in (0, 1):
        color, depth, vel, hist, prev = ts = [moved(t, by) for t in images]
        screen, new = torch.zeros_like(hist), torch.zeros_like(hist)
        at = lambda t: t.data_ptr() + by * t.element_size()
        img = FrameImages()
        img.color, img.depth, img.velocity, img.history, img.history_depth = [at(t) for t in ts]
        img.result_history, img.result_screen = at(new), at(screen)
        img.width, img.height, img.pitch = W, H, W
        img.input_width, img.input_height, img.input_pitch = lo[0], lo[1], lo[0]
        img.color_format, img.velocity_format = fmt, w["vel"]
        check(lib().taa_resolve_frame(C.byref(U), C.byref(img), C.byref(K), arith, None))
        torch.cuda.synchronize()
        out.append((screen[by:], new[by:]))
    assert_same_bits(out[0][0], out[1][0], "screen")
    assert_same_bits(out[0][1], out[1][1], "history")
