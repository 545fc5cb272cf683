"""Conv2d shapes of the gathered-window kernel at the sizes where it can go
wrong: one pixel past and short of a tile, tiles that cross images, channel
tiles and K blocks that are not whole, padding wider than the window, outputs
whose planes are no multiple of 4 pixels, every stored type.

The bar is derived: the operands are known exactly (x rounded to bf16, the
weights' decoded values), so only the fp32 sums differ from fp64, by at most
K * 2^-23 times the sum of |products|."""
import numpy as np
import pytest
import torch

import oracle as O
from novann_amd import functional as F
from novann_amd import quant
from novann_amd.module import Parameters, QuantizedParameters
from oracle import functional_ref as R
from tests.gpu_util import bf16_round

pytestmark = pytest.mark.gpu

# (N, C, H, W, C_out, k, stride, padding)
SHAPES = [
    (1, 16, 8, 8, 16, 1, 1, 0),       # 64 pixels: one tile; K = 16
    (1, 8, 5, 13, 17, 3, 1, 1),       # 65 pixels, 17 channels, K = 72
    (9, 70, 7, 7, 33, 3, 1, 1),       # tiles across images, K = 630
    (3, 66, 9, 7, 129, 3, 2, 1),      # strided, 8-tile channel block and one more
    (2, 40, 15, 11, 65, 5, 3, 4),     # stride 3, padding near the window's size
    (1, 3, 12, 10, 5, 5, 2, 6),       # padding wider than the window
    (70, 80, 1, 1, 12, 1, 1, 0),      # one pixel an image
    (520, 68, 6, 6, 70, 3, 1, 1),     # neighbouring pixel tiles a wave, last one ragged
]


def reference(x, w, stride, pad, bias=None):
    return R.conv2d(x.astype(np.float64), w.astype(np.float64), (stride, stride), (pad, pad),
                    "zeros", bias)


def check(got, x, w, stride, pad, what):
    want = reference(x, w, stride, pad)
    bound = max(w[0].size, 8) * 2.0**-23 * reference(np.abs(x), np.abs(w), stride, pad) + 1e-30
    assert got.shape == want.shape
    assert np.all(np.abs(got.astype(np.float64) - want) <= bound), what


def make(shape, wdt):
    n, c, h, w, co, k, s, p = shape
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    wt = (rng.standard_normal((co, c, k, k)) * 0.1).astype(np.float32)
    if wdt in ("f32", "bf16"):
        q = Parameters(torch.from_numpy(wt if wdt == "f32" else bf16_round(wt)).cuda())
        return x, q, bf16_round(wt)
    q = QuantizedParameters.from_float(wt, wdt)
    return x, q, q.dequantize().cpu().numpy()


@pytest.mark.parametrize("wdt", ["e4m3", "e2m1", "f32"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16, torch.float16])
def test_gathered_conv_exact_operands(shape, wdt, xdt):
    print(f"gathered conv {shape} {wdt} {xdt}", flush=True)
    x, q, w = make(shape, wdt)
    xd = torch.from_numpy(x).cuda().to(xdt)
    y = F.conv2d(xd, q, shape[5], shape[6], shape[7]).cpu().numpy()
    check(y, bf16_round(xd.float().cpu().numpy()), w, shape[6], shape[7], shape)


@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[3]], ids=["65px", "strided"])
def test_gathered_conv_fp8_input(shape):
    x, q, w = make(shape, "e5m2")
    xq = quant.quantize(torch.from_numpy(x).cuda(), "e4m3")
    y = F.conv2d(xq, q, shape[5], shape[6], shape[7]).cpu().numpy()
    xv = quant.dequantize(xq).cpu().numpy()
    # the scale is applied after the sums: one more rounding
    want = reference(xv, w, shape[6], shape[7])
    bound = (w[0].size + 2) * 2.0**-23 * reference(np.abs(xv), np.abs(w), shape[6], shape[7])
    assert np.all(np.abs(y.astype(np.float64) - want) <= bound + 1e-30)


@pytest.mark.parametrize("out", ["bf16", "e4m3"])
@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[2], SHAPES[7]], ids=["65px", "7x7", "many"])
def test_gathered_conv_epilogue(shape, out):
    """The fused epilogue equals its steps on the plain output bit for bit."""
    x, q, _ = make(shape, "e4m3")
    xd = torch.from_numpy(x).cuda()
    rng = np.random.default_rng(3)
    mul, add = (rng.standard_normal(shape[4]).astype(np.float32) for _ in range(2))
    amax = torch.zeros(1, device="cuda")
    y = F.conv2d(xd, q, *shape[5:]).cpu().numpy()
    got = F.conv2d(xd, q, *shape[5:], epilogue=F.Epilogue(
        channel_mul=mul, channel_add=add, relu=True, out_dtype=out, out_amax=amax))
    v = y * mul.reshape(1, -1, 1, 1) + add.reshape(1, -1, 1, 1)
    v = (v * (v > 0)).astype(np.float32)
    code = {"bf16": O.BF16, "e4m3": O.E4M3}[out]
    want = O.cast(v.reshape(-1), O.F32, code)
    data = got.data if out == "e4m3" else got.reshape(-1)
    raw = data.view(torch.uint8 if out == "e4m3" else torch.int16).cpu().numpy()
    assert np.array_equal(raw.view(want.dtype).reshape(-1), want)
    assert float(amax) == np.abs(v).max()
