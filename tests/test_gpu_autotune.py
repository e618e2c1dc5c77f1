"""The autotuner runs the kernel its class's frames run: every storage and arithmetic, and a tuned class resolves to the
bits of an untuned one."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from gpu_helpers import assert_same_bits  # noqa: E402
from test_gpu_upscale import inputs  # noqa: E402
from taastar import (ARITH_FP16, ARITH_FP32, FMT_RGBA16F, FMT_RGBA32F, VEL_RG16F, VEL_RG32F, FrameImages, check, lib)  # noqa: E402
from taastar.workloads import cas_for, uniforms_for, workload  # noqa: E402


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("W,H", [(325, 181), (1283, 721)])
@pytest.mark.parametrize("cas", [True, False])
@pytest.mark.parametrize("fmt,arith", [(FMT_RGBA16F, ARITH_FP16), (FMT_RGBA16F, ARITH_FP32), (FMT_RGBA32F, ARITH_FP16), (FMT_RGBA32F, ARITH_FP32)])
def test_autotune(W, H, cas, fmt, arith):
    print(f"case autotune {W}x{H} cas {cas} fmt {fmt} arith {arith}", flush=True)
    w = workload("c2", fmt=fmt, vel=VEL_RG16F if fmt == FMT_RGBA16F else VEL_RG32F)
    color, depth, vel, hist, prev = inputs(W, H, W, H, W, W, fmt, 3, False, 17)
    U = uniforms_for(w, 1, (0.2 / W, 0.1 / H))
    K = cas_for(w, W, H) if cas else None

    def resolve():
        screen, new = torch.zeros_like(hist), torch.zeros_like(hist)
        img = FrameImages()
        img.color, img.depth, img.velocity = color.data_ptr(), depth.data_ptr(), vel.data_ptr()
        img.history, img.history_depth = hist.data_ptr(), prev.data_ptr()
        img.result_history, img.result_screen = new.data_ptr(), screen.data_ptr()
        img.width, img.height, img.pitch = W, H, W
        img.color_format, img.velocity_format = fmt, w["vel"]
        check(lib().taa_resolve_frame(C.byref(U), C.byref(img), C.byref(K) if K else None, arith, None))
        torch.cuda.synchronize()
        return screen, new

    before = resolve()
    ctx, best, us = C.c_void_p(), C.c_int32(-1), C.c_float()
    check(lib().taa_ctx_create(0, 0, C.byref(ctx)))
    try:
        check(lib().taa_autotune(ctx, W, H, fmt, arith, int(cas), 3, C.byref(best), C.byref(us)))
        assert 0 <= best.value < lib().taa_tile_shape_count() and us.value > 0.0
        after = resolve()
    finally:
        check(lib().taa_tile_shape_select(W, H, fmt, arith, int(cas), -1))
        check(lib().taa_ctx_destroy(ctx))
    assert_same_bits(before[0], after[0], "screen")
    assert_same_bits(before[1], after[1], "history")
