"""Conv2d with the input staged in chunks of 32 channels, at the sizes where it
can go wrong: bands that do not divide the output rows, bands whose input rows
are all padding, a last group of fewer images, channel blocks that are not
whole, output planes that are no multiple of 4 pixels, one to three chunks,
rows of the least width, each tile, both windows, every stored type.

The bar is derived: the operands are known exactly (x rounded to bf16, the
weights' decoded values), so only the fp32 sums differ from fp64, by at most
K * 2^-23 times the sum of |products|."""
import numpy as np
import pytest
import torch

import oracle as O
from novann_amd import functional as F
from novann_amd import quant
from tests.gpu_util import bf16_round
from tests.test_gpu_conv2d_gather import check, make, reference

pytestmark = pytest.mark.gpu

# (N, C, H, W, C_out, k, stride, padding)
SHAPES = [
    (65, 32, 7, 7, 33, 3, 1, 1),       # 2 images a workgroup, the last alone; 49 pixels
    (33, 64, 6, 6, 65, 3, 1, 1),       # runs of 4 pixels, 3 images, one channel past a block
    (40, 96, 13, 11, 31, 3, 1, 1),     # 3 chunks, 256-pixel tile, uneven last band
    (34, 32, 14, 14, 1, 3, 1, 0),      # one channel, no padding
    (4, 32, 12, 124, 40, 3, 1, 3),     # one row a band; first and last rows all padding
    (12, 64, 29, 31, 129, 3, 2, 1),    # strided, 128-channel block and one more
    (48, 32, 17, 13, 70, 3, 3, 2),     # stride 3, too few workgroups for the wide tile
    (520, 32, 4, 4, 64, 3, 1, 1),      # rows of the least width, 8 images
    (36, 64, 9, 15, 66, 1, 1, 0),      # 1 x 1
    (40, 96, 15, 14, 20, 1, 2, 1),     # 1 x 1, strided, padded, 256-pixel tile
]


@pytest.mark.parametrize("wdt", ["e4m3", "e2m1"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16, torch.float16])
def test_chunked_conv_exact_operands(shape, wdt, xdt):
    print(f"chunked conv {shape} {wdt} {xdt}", flush=True)
    x, q, w = make(shape, wdt)
    xd = torch.from_numpy(x).cuda().to(xdt)
    y = F.conv2d(xd, q, shape[5], shape[6], shape[7]).cpu().numpy()
    check(y, bf16_round(xd.float().cpu().numpy()), w, shape[6], shape[7], shape)


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[5]], ids=["7x7", "strided"])
def test_chunked_conv_fp8_input(shape):
    x, q, w = make(shape, "e5m2")
    xq = quant.quantize(torch.from_numpy(x).cuda(), "e4m3")
    y = F.conv2d(xq, q, shape[5], shape[6], shape[7]).cpu().numpy()
    xv = quant.dequantize(xq).cpu().numpy()
    # the scale is applied after the sums: one more rounding
    want = reference(xv, w, shape[6], shape[7])
    bound = (w[0].size + 2) * 2.0**-23 * reference(np.abs(xv), np.abs(w), shape[6], shape[7])
    assert np.all(np.abs(y.astype(np.float64) - want) <= bound + 1e-30)


@pytest.mark.parametrize("out", ["bf16", "e4m3"])
@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[1], SHAPES[2]], ids=["7x7", "6x6", "bands"])
def test_chunked_conv_epilogue(shape, out):
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


def test_chunked_conv_nan_stays_in_its_windows():
    """A NaN pixel reaches the outputs whose windows hold it and no other."""
    shape = SHAPES[1]
    x, q, _ = make(shape, "e4m3")
    x[2, 40, 5, 0] = np.nan
    y = F.conv2d(torch.from_numpy(x).cuda(), q, 3, 1, 1).cpu().numpy()
    bad = np.zeros(y.shape, bool)
    bad[2, :, 4:6, 0:2] = True
    assert np.array_equal(np.isnan(y), bad)


# (N, C, H, W, C_out, k, stride, padding): 32 or 64 channels that chunks, bands
# and the gathered kernel all take, each side of the lines between them
BETWEEN = [
    (256, 32, 7, 7, 32, 3, 1, 1), (600, 32, 7, 7, 17, 3, 1, 1), (64, 64, 9, 9, 30, 3, 1, 1),
    (256, 64, 7, 7, 32, 1, 1, 0), (600, 32, 9, 9, 64, 1, 1, 0), (40, 32, 14, 14, 32, 3, 2, 1),
    (90, 64, 10, 9, 33, 3, 2, 1), (300, 32, 9, 9, 70, 3, 1, 1), (520, 32, 12, 12, 70, 3, 1, 1),
    (3, 32, 99, 100, 96, 3, 1, 1), (512, 32, 13, 13, 96, 3, 1, 1), (200, 32, 28, 28, 48, 1, 1, 0),
]


@pytest.mark.parametrize("wdt", ["e4m3", "e2m1"])
@pytest.mark.parametrize("shape", BETWEEN, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16])
def test_shapes_that_several_kernels_take(shape, wdt, xdt):
    test_chunked_conv_exact_operands(shape, wdt, xdt)
