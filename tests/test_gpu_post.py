"""Edge AA and the stand-alone CAS against the oracle, bit for bit in the storage format, at the edges of their waves:
64 or 128 columns, one row a wave or four, ragged both ways, padded rows untouched."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from test_gpu_edge_aa import bits, consts, run, stored  # noqa: E402
from taastar import FMT_RGBA16F, FMT_RGBA32F, check, lib  # noqa: E402
from taastar.device import color_dtype  # noqa: E402
from taastar.workloads import cas_for, encode_color, workload  # noqa: E402


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


# 512 tiles of 16 rows take four rows a wave: the last two sizes
@pytest.mark.parametrize("W,H", [(1, 3), (2, 1), (63, 5), (64, 4), (65, 6), (127, 3), (128, 9), (129, 2), (257, 4099), (1151, 913)])
@pytest.mark.parametrize("fmt", [FMT_RGBA32F, FMT_RGBA16F])
@pytest.mark.parametrize("pad", [0, 3])
def test_rows_and_columns(oracle, W, H, fmt, pad):
    print(f"case post {W}x{H} fmt {fmt} pad {pad}", flush=True)
    rng = np.random.default_rng(W * 10007 + H)
    src = encode_color(np.concatenate([rng.uniform(0, 1, (H, W, 3)) ** 2, np.ones((H, W, 1))], -1).astype(np.float32), fmt)
    mask = rng.integers(0, 3, (H, W)).astype(np.uint32)
    k = consts(W, H)
    got = run(src, mask, fmt, k, pad)
    ref = stored(oracle.edge_aa(src.astype(np.float32), mask, k.subpix, k.edge_threshold, k.edge_threshold_min), fmt)
    assert np.count_nonzero(bits(got[:, :W]) != bits(ref)) == 0, "edge AA"
    assert np.all(got[:, W:] == 7.0), "edge AA: row padding written"

    K = cas_for(workload("c2"), W, H)
    s = torch.full((H, W + pad, 4), float("nan"), dtype=color_dtype(fmt), device="cuda")
    s[:, :W] = torch.from_numpy(src).cuda()
    d = torch.full_like(s, 7.0)
    check(lib().taa_cas_apply(C.c_void_p(s.data_ptr()), C.c_void_p(d.data_ptr()), W, H, W + pad, fmt, C.byref(K), None))
    torch.cuda.synchronize()
    got = d.cpu().numpy()
    ref = stored(oracle.cas(src.astype(np.float32), K.const1[0]), fmt)
    assert np.count_nonzero(bits(got[:, :W]) != bits(ref)) == 0, "CAS"
    assert np.all(got[:, W:] == 7.0), "CAS: row padding written"
