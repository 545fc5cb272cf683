"""Linear products on the kernels of 128-row tiles, which run where 128 x 256
tiles cover more than an eighth of the CUs: the ping-pong kernel (FP8 W), the
wide-K kernel (FP4 W) and the staged-decode kernel (16-bit W, and whole tiles
that the other two do not have), in whole tiles.

The bar is derived: the operands the MFMAs multiply are known exactly, so only
the fp32 sums differ from fp64, by at most K * 2^-23 times the sum of
|products|, and the scale, applied after them, adds a rounding."""
import numpy as np
import pytest
import torch

from tests.gpu_util import bf16_round
from tests.test_gpu_epilogue import linear_x, quantized_codes, x_codes

pytestmark = pytest.mark.gpu


def takes_tiles(m, n):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    return -(-m // 128) * -(-n // 256) > cus // 8


# (M, K, N): the staged-decode kernel at both tile widths -- one K block and
# several, K and columns that are no multiple of the other kernels' 128 and 256
STAGED = [(1024, 64, 2304), (1152, 320, 1280), (2048, 64, 640), (2176, 192, 384),
          (2048, 128, 1152)]


@pytest.mark.parametrize("wdt", ["e4m3", "e5m2", "e2m1", "bf16", "f16"])
@pytest.mark.parametrize("m,k,n", STAGED)
def test_staged_tiles_exact_operands(m, k, n, wdt):
    assert takes_tiles(m, n)
    rng = np.random.default_rng(m + k + n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    w = (rng.standard_normal((n, k)) * 0.1).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    wd, ws, wdeq = quantized_codes(w, wdt, rng)
    for xt in ("f32", "bf16", "f16", "e4m3", "e5m2"):
        print(f"staged tiles {wdt} x {xt} {m}x{k}x{n}", flush=True)
        if xt == "f32":
            xd, sx, xv = torch.from_numpy(x).cuda(), None, x
        else:
            xd, sx, xv = x_codes(x, xt)
        y = linear_x(xd, xt, sx, m, k, wd, wdt, ws, n, bias).view(np.float32)
        s = 1.0 if sx is None else float(sx)
        # the operands multiplied: x rounded to bf16, W's codes (a 16-bit W
        # rounded to bf16)
        a = bf16_round(xv).astype(np.float64) * s
        b = (wdeq if ws is not None else bf16_round(wdeq)).astype(np.float64).T
        size = np.abs(a) @ np.abs(b)
        bound = (k + 3) * 2.0**-23 * size + 2.0**-23 * np.abs(bias) + 1e-30
        assert np.all(np.abs(y.astype(np.float64) - (a @ b + bias)) <= bound), xt
