"""The FP16-storage throughput kernel's variants (rows a thread, history window or direct gather, fixed or read
options): each against the oracle at the edges of its regions, and all the same bits."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from gpu_helpers import Sequence, assert_same_bits, psnr, rel_err  # noqa: E402
from test_gpu_edges import assert_fp16_indices  # noqa: E402
from taastar import (ARITH_FP16, FMT_RGBA16F, KERNEL_FP16, VEL_RG16F, VEL_RGBA16F, check, default_params, lib)  # noqa: E402
from taastar.workloads import workload  # noqa: E402


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


class Forced:
    """The class's table entry, which selects the rows a thread (entry 0: one, 1: two, 2: four)."""

    def __init__(self, W, H, cas, index):
        self.key, self.index = (W, H, FMT_RGBA16F, ARITH_FP16, int(cas)), index

    def __enter__(self):
        check(lib().taa_tile_shape_select(*self.key, self.index))

    def __exit__(self, *exc):
        check(lib().taa_tile_shape_select(*self.key, -1))


def scattered(seq, motion, seed):
    """Displace blocks of the velocity field by up to `motion` texels, so that a region's footprints spread."""
    rng = np.random.default_rng(seed)
    render = seq.scene.render

    def spread(frame, threads=0):
        c, d, v4, jit = render(frame, threads)
        v = v4.copy()
        H, W = v.shape[:2]
        by, bx = rng.uniform(-motion, motion, ((H + 10) // 11, (W + 12) // 13)), rng.uniform(-motion, motion, ((H + 10) // 11, (W + 12) // 13))
        v[..., 0] += np.kron(bx, np.ones((11, 13)))[:H, :W] / W
        v[..., 1] += np.kron(by, np.ones((11, 13)))[:H, :W] / H
        return c, d, v.astype(np.float32), jit

    seq.scene.render = spread


# widths and heights on both sides of 30 / 32 columns and 14 / 16 / 30 / 32 rows, one and two regions; motion within
# the window's margin (0, 6 texels) and beyond it (40)
@pytest.mark.parametrize("W,H,motion", [(33, 31, 0), (61, 29, 6), (95, 71, 6), (127, 65, 40), (3, 40, 6)])
@pytest.mark.parametrize("cas", [True, False])
def test_variants_against_the_oracle(oracle, W, H, motion, cas):
    kept = []
    for index in (0, 1, 2):
        print(f"case {W}x{H} motion {motion} cas {cas} entry {index}", flush=True)
        with Forced(W, H, cas, index):
            seq = Sequence(workload("c2", fmt=FMT_RGBA16F, vel=VEL_RG16F), width=W, height=H, cas=cas, arith=ARITH_FP16, debug=False, shipped=True)
            scattered(seq, motion, 11)
            assert seq.kernel()[0] == KERNEL_FP16
            for _ in range(3):
                out = seq.step(oracle)
                assert_fp16_indices(out)
                # the bars of the small-size FP16 tests
                if cas:
                    assert psnr(out["gpu_screen"][..., :3], out["oracle_screen"][..., :3]) > 55.0
                else:
                    e = rel_err(out["gpu_history"][..., :3], out["oracle_history"][..., :3], floor=1e-2)
                    assert np.quantile(e, 0.999) < 1e-2
            kept.append((seq.ship.screen.clone(), seq.ship.hist_in.clone()))
    for s, h in kept[1:]:
        assert_same_bits(s, kept[0][0], "screen")
        assert_same_bits(h, kept[0][1], "history")


@pytest.mark.parametrize("index", [0, 1, 2])
@pytest.mark.parametrize("preset", ["defaults", "production"])
def test_fixed_options_equal_read_ones(index, preset):
    """The forms with every option fixed write the bits of the form that reads its options (which a parameter without
    effect here, or a bound debug image, selects)."""
    W, H = 95, 61
    rgba = preset == "defaults"
    p = default_params() if rgba else workload("c2")["params"]()
    w = workload("c2", fmt=FMT_RGBA16F, vel=VEL_RGBA16F if rgba else VEL_RG16F)
    out = []
    with Forced(W, H, True, index):
        for other in (False, True):
            q = type(p).from_buffer_copy(p)
            if other and not rgba:
                q.mVelBasedAlpha, q.mVelBasedAlphaFactor, q.mVelBasedAlphaMax = 1, 0.0, 0.0  # Lottes replaces alpha
            print(f"case {preset} entry {index} other {other}", flush=True)
            seq = Sequence(w, width=W, height=H, cas=True, arith=ARITH_FP16, params=q, debug=other and rgba)
            seq.bufs.inspect = None
            for f in range(3):
                col, dep, vel4, jit = seq.scene.render(f)
                from taastar.workloads import encode_color, encode_velocity, uniforms_for
                seq.bufs.upload(encode_color(col, w["fmt"]), dep, encode_velocity(vel4, w["vel"]))
                seq.bufs.resolve(uniforms_for(w, f, jit, params=q), seq.cas, ARITH_FP16)
            torch.cuda.synchronize()
            out.append((seq.bufs.screen.clone(), seq.bufs.hist_in.clone()))
    assert_same_bits(out[0][0], out[1][0], "screen")
    assert_same_bits(out[0][1], out[1][1], "history")
