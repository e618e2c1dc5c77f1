"""The exact kernel of the production feature set against the general form (which a bound debug image selects): the same
bits, single frames and batches, on both sides of the line that selects it."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from gpu_helpers import assert_same_bits  # noqa: E402
from test_gpu_upscale import inputs, test_batches_equal_sessions_alone as batches  # noqa: E402
from taastar import ARITH_FP32, FMT_RGBA16F, FMT_RGBA32F, VEL_RG16F, VEL_RG32F, FrameImages, check, lib  # noqa: E402
from taastar.workloads import cas_for, uniforms_for, workload  # noqa: E402


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


# regions are 30 x 14 (CAS) or 32 x 16 texels, 900 to 1500 of them select the kernel; the second size is a texel beyond
# whole regions, the last columns and rows of the third are one texel of a region; motion within the window and beyond it
@pytest.mark.parametrize("W,H,motion,odd", [(960, 540, 0, False), (1441, 897, 6, True), (961, 1121, 6, True), (1280, 720, 60, False),
                                            (3, 24001, 4, False), (24001, 3, 4, True), (333, 111, 6, True)])
@pytest.mark.parametrize("fmt", [FMT_RGBA16F, FMT_RGBA32F])
def test_equals_the_general_form(W, H, motion, odd, fmt):
    for k, (cas, pad, reset, split) in enumerate([(True, 0, 0, 0), (False, 3, 0, 0), (True, 5, 0, W // 3), (True, 0, 1, 0)]):
        print(f"case {W}x{H} fmt {fmt} cas {cas} pad {pad} reset {reset} split {split}", flush=True)
        pitch = W + pad
        color, depth, vel, hist, prev = inputs(W, H, W, H, pitch, pitch, fmt, motion, odd, 71 + k)
        w = workload("c2", fmt=fmt, vel=VEL_RG16F if fmt == FMT_RGBA16F else VEL_RG32F)
        U = uniforms_for(w, 1, (0.3 / W, -0.4 / H))
        U.mResetHistory, U.splitScreen, U.splitX = reset, int(split > 0), split
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
            img.color_format, img.velocity_format = fmt, w["vel"]
            check(lib().taa_resolve_frame(C.byref(U), C.byref(img), C.byref(K) if K else None, ARITH_FP32, None))
            torch.cuda.synchronize()
            out.append((screen, new))
        assert_same_bits(out[0][0], out[1][0], "screen")
        assert_same_bits(out[0][1], out[1][1], "history")


@pytest.mark.parametrize("specs", [[((480, 270), (480, 270)), ((640, 361), (640, 361)), ((33, 65), (33, 65))],
                                   [((160, 90), (160, 90)), ((95, 61), (95, 61))]])
@pytest.mark.parametrize("fmt", [FMT_RGBA16F, FMT_RGBA32F])
def test_batches(specs, fmt):
    batches(specs, fmt, ARITH_FP32)
