"""The upsampling kernel of the production feature set against the general form (which a bound debug image selects): the
same bits at the edges of its tiles, over scales on both sides of the line that selects it, and in batches."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from gpu_helpers import assert_same_bits  # noqa: E402
from taastar import (ARITH_FP16, ARITH_FP32, FMT_RGBA16F, FMT_RGBA32F, VEL_RG16F, VEL_RG32F, BatchItem, FrameImages, SessionIO,  # noqa: E402
                     Uniforms, check, lib)
from taastar.device import color_dtype  # noqa: E402
from taastar.workloads import cas_for, uniforms_for, workload  # noqa: E402


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def inputs(Wl, Hl, W, H, pl, pitch, fmt, motion, odd, seed):
    """Random images; blocks of velocity up to `motion` output texels; `odd`: infinities, NaN and -0 among them."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.rand(*s, generator=g, device="cuda")
    color, hist = r(Hl, pl, 4) ** 3 * 4, r(H, pitch, 4) ** 3 * 4
    depth, prev = 0.9 + 0.1 * r(Hl, pl), 0.9 + 0.1 * r(Hl, pl)
    prev[: Hl // 2] = depth[: Hl // 2]  # no rejection in the upper half
    blocks = ((r((Hl + 8) // 9, (pl + 10) // 11, 2) - 0.5) * 2 * motion).repeat_interleave(9, 0).repeat_interleave(11, 1)[:Hl, :pl]
    vel = blocks / torch.tensor([W, H], device="cuda")
    if odd:
        bad = torch.tensor([float("inf"), -float("inf"), float("nan"), -0.0, 0.0, 1e30, 1e-42], device="cuda")
        for t in (color, hist, depth, prev, vel):
            f = t.view(-1)
            at = torch.randint(0, f.numel(), (max(8, f.numel() // 200),), generator=g, device="cuda")
            f[at] = bad[torch.randint(0, len(bad), at.shape, generator=g, device="cuda")]
    cd = color_dtype(fmt)
    return color.to(cd), depth, vel.to(cd).contiguous(), hist.to(cd), prev


# tiles are 30 x 14 / 30 x 30 (CAS) or 32 x 16 / 32 x 32 output texels: one, two and many of them, ragged; the last case has
# enough for the four-row tile
@pytest.mark.parametrize("lo,hi,motion,odd", [
    ((3, 2), (7, 5), 2, False), ((16, 8), (33, 17), 0, False), ((61, 29), (92, 57), 6, True), ((50, 70), (101, 141), 40, False),
    ((64, 64), (70, 64), 6, False), ((43, 90), (130, 91), 6, True), ((481, 301), (1441, 901), 6, True)])
@pytest.mark.parametrize("fmt,arith", [(FMT_RGBA16F, ARITH_FP16), (FMT_RGBA16F, ARITH_FP32), (FMT_RGBA32F, ARITH_FP16), (FMT_RGBA32F, ARITH_FP32)])
def test_equals_the_general_form(lo, hi, motion, odd, fmt, arith):
    (Wl, Hl), (W, H) = lo, hi
    for k, (cas, upsampling, pad, reset) in enumerate([(True, True, 0, 0), (False, True, 5, 0), (True, False, 3, 0), (True, True, 1, 1)]):
        print(f"case {lo} -> {hi} fmt {fmt} arith {arith} cas {cas} upsampling {upsampling} pad {pad} reset {reset}", flush=True)
        pl, pitch = Wl + pad, W + 2 * pad
        color, depth, vel, hist, prev = inputs(Wl, Hl, W, H, pl, pitch, fmt, motion, odd, 31 + k)
        w = workload("c2", fmt=fmt, vel=VEL_RG16F if fmt == FMT_RGBA16F else VEL_RG32F)
        U = uniforms_for(w, 1, (0.3 / Wl, -0.4 / Hl))
        U.mUpsampling, U.mResetHistory = int(upsampling), reset
        K = cas_for(w, W, H) if cas else None
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
            img.input_width, img.input_height, img.input_pitch = Wl, Hl, pl
            img.color_format, img.velocity_format = fmt, w["vel"]
            check(lib().taa_resolve_frame(C.byref(U), C.byref(img), C.byref(K) if K else None, arith, None))
            torch.cuda.synchronize()
            out.append((screen, new))
        assert_same_bits(out[0][0], out[1][0], "screen")
        assert_same_bits(out[0][1], out[1][1], "history")


@pytest.mark.parametrize("specs", [[((96, 54), (192, 108)), ((64, 40), (200, 91))],
                                   [((96, 54), (192, 108)), ((150, 80), (160, 90))],  # one below the line: the general kernel
                                   [((33, 20), (65, 41)), ((64, 40), (64, 40)), ((480, 300), (1441, 901))]])
@pytest.mark.parametrize("fmt,arith", [(FMT_RGBA16F, ARITH_FP16), (FMT_RGBA32F, ARITH_FP32)])
def test_batches_equal_sessions_alone(specs, fmt, arith):
    w = workload("c2", fmt=fmt, vel=VEL_RG16F if fmt == FMT_RGBA16F else VEL_RG32F)
    memcpy = lib().hipMemcpy
    memcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]

    def run(batch):
        ctx, sess, scrs, Us, Ks = C.c_void_p(), [], [], [], []
        check(lib().taa_ctx_create(0, 0, C.byref(ctx)))
        items = (BatchItem * len(specs))()
        for k, ((Wl, Hl), (W, H)) in enumerate(specs):
            s = C.c_void_p()
            check(lib().taa_session_open_scaled(ctx, W, H, Wl, Hl, fmt, w["vel"], C.byref(s)))
            sess.append(s)
            scrs.append(torch.zeros(H, W, 4, dtype=color_dtype(fmt), device="cuda"))
            Us.append(Uniforms())
            Ks.append(cas_for(w, W, H))
            items[k].session, items[k].uniforms = s, C.pointer(Us[k])
            items[k].cas, items[k].result_screen = C.pointer(Ks[k]), scrs[k].data_ptr()
        got = []
        for f in range(3):
            for k, ((Wl, Hl), (W, H)) in enumerate(specs):
                io = SessionIO()
                check(lib().taa_session_io(sess[k], C.byref(io)))
                assert (io.width, io.height, io.pitch) == (Wl, Hl, Wl)
                color, depth, vel, _, _ = inputs(Wl, Hl, W, H, Wl, W, fmt, 5, False, 100 * f + k)
                torch.cuda.synchronize()
                for ptr, t in ((io.color, color), (io.depth, depth), (io.velocity, vel)):
                    assert memcpy(C.c_void_p(ptr), C.c_void_p(t.data_ptr()), t.numel() * t.element_size(), 3) == 0
                U = uniforms_for(w, f, (0.2 / Wl, 0.1 / Hl))
                U.mUpsampling = int((Wl, Hl) != (W, H))
                C.memmove(C.addressof(Us[k]), C.addressof(U), C.sizeof(Uniforms))
            if batch:
                check(lib().taa_batch_submit(ctx, len(specs), items, arith, None))
            else:
                for k in range(len(specs)):
                    check(lib().taa_session_resolve(sess[k], C.byref(Us[k]), C.byref(Ks[k]), C.c_void_p(scrs[k].data_ptr()), arith, None))
            torch.cuda.synchronize()
            got.append([t.clone() for t in scrs])
        for s in sess:
            check(lib().taa_session_close(s))
        check(lib().taa_ctx_destroy(ctx))
        return got

    print(f"case batch {specs} fmt {fmt}", flush=True)
    alone, batch = run(False), run(True)
    for f in range(3):
        for k in range(len(specs)):
            assert_same_bits(alone[f][k], batch[f][k], f"frame {f} session {k}")
