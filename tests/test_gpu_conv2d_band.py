"""The band convolution at sizes that are dispatched to it (zero padding runs in
bands from as many of them as there are CUs, or with many pixels in few): its
3 x 3 kernel with constant regrouping of the weights and its general one, whole
and partial blocks of output channels, narrow outputs staged through LDS and
stored by the lanes, amax and the fused epilogue, and every stored x."""
import numpy as np
import pytest
import torch

import oracle as O
from oracle import functional_ref as R
from tests.gpu_util import bf16_round
from tests.test_gpu_epilogue import (Epi, check_all_outputs, combined_scale, conv_ex, conv_x,
                                     quantized_codes, rounding_classes, x_codes)

pytestmark = pytest.mark.gpu

# wdt, (N, C, H, W), C_out, (KH, KW), pad: at least one band a CU, and channels
# that are no multiple of 32 (those of 32 have another kernel)
CASES = [
    ("e2m1", (72, 16, 28, 28), 48, (3, 3), (1, 1)),   # 4 bands an image, 3 x 3 regrouping
    ("e4m3", (300, 24, 12, 12), 20, (3, 3), (1, 1)),  # one band an image
    ("e5m2", (130, 8, 14, 14), 70, (3, 3), (1, 1)),   # two blocks of output channels
    ("e4m3", (260, 40, 9, 11), 33, (3, 3), (1, 1)),   # rows of no whole 4 columns
    ("bf16", (258, 6, 10, 12), 18, (3, 3), (0, 1)),   # the general kernel: 16-bit weights
    ("e2m1", (257, 5, 12, 8), 16, (2, 5), (1, 2)),    # and another window
    ("e4m3", (60, 16, 22, 24), 48, (3, 3), (1, 1)),   # fewer bands than CUs, many pixels
]


@pytest.mark.parametrize("wdt,xs,C_out,k,pad", CASES)
def test_bands_exact_operands_and_epilogue(wdt, xs, C_out, k, pad):
    print(f"bands {wdt} {xs} -> {C_out} k={k} p={pad}", flush=True)
    rng = np.random.default_rng(sum(xs) + C_out)
    x = rng.standard_normal(xs).astype(np.float32)
    wshape = (C_out, xs[1]) + k
    w = (rng.standard_normal(wshape) * 0.1).astype(np.float32)
    bias = rng.standard_normal(C_out).astype(np.float32)
    wd, ws, wdeq = quantized_codes(w, wdt, rng)
    y0 = conv_ex(x, wd, wdt, ws, wshape, (1, 1), pad, "zeros", None, bias)
    # only the fp32 sums, the scale and the bias round: K + 2 roundings
    xb, w64 = bf16_round(x).astype(np.float64), wdeq.astype(np.float64)
    want = R.conv2d(xb, w64, (1, 1), pad, "zeros", bias.astype(np.float64))
    size = R.conv2d(np.abs(xb), np.abs(w64), (1, 1), pad, "zeros",
                    np.abs(bias).astype(np.float64))
    K = xs[1] * k[0] * k[1]
    assert np.all(np.abs(y0.view(np.float32) - want) <= (K + 2) * 2.0**-23 * size + 1e-30)
    check_all_outputs(lambda ep: conv_ex(x, wd, wdt, ws, wshape, (1, 1), pad, "zeros", ep, bias),
                      y0, C_out, rng)


@pytest.mark.parametrize("xt", ["bf16", "f16", "e4m3", "e5m2"])
@pytest.mark.parametrize("wdt,xs,C_out,k,pad", [CASES[0], CASES[3], CASES[4]])
def test_bands_read_stored_activations(xt, wdt, xs, C_out, k, pad):
    rng = np.random.default_rng(sum(xs) * 3 + C_out)
    x = rng.standard_normal(xs).astype(np.float32)
    wshape = (C_out, xs[1]) + k
    w = (rng.standard_normal(wshape) * 0.1).astype(np.float32)
    bias = rng.standard_normal(C_out).astype(np.float32)
    wd, ws, _ = quantized_codes(w, wdt, rng)
    xd, sx, xdec = x_codes(x, xt)
    got = conv_x(xd, xt, sx, xs, wd, wdt, ws, wshape, (1, 1), pad, "zeros", bias)
    want = conv_x(torch.from_numpy(np.ascontiguousarray(xdec)).cuda(), "f32", None, xs, wd, wdt,
                  combined_scale(ws, sx), wshape, (1, 1), pad, "zeros", bias)
    assert np.array_equal(got, want)


def test_staged_bf16_stores_round_every_class():
    """With x = 0 each output channel is its bias, so the bias vector feeds the
    encoder of the stores that leave through LDS every rounding class."""
    rng = np.random.default_rng(17)
    bias = rounding_classes(rng)
    C_out, C, n = bias.size, 8, 8
    x = np.zeros((n, C, 4, 4), np.float32)
    w = rng.standard_normal((C_out, C, 1, 1)).astype(np.float32)
    wd, ws, _ = quantized_codes(w, "e4m3", rng)
    assert n * -(-C_out // 64) >= torch.cuda.get_device_properties(0).multi_processor_count
    y0 = conv_ex(x, wd, "e4m3", ws, w.shape, (1, 1), (0, 0), "zeros", None, bias)
    ep = Epi(C_out, rng, relu=False, out="bf16", amax=False, mul=False, add=False)
    got = conv_ex(x, wd, "e4m3", ws, w.shape, (1, 1), (0, 0), "zeros", ep, bias).reshape(-1)
    assert np.array_equal(got, O.cast(y0.view(np.float32).reshape(-1), O.F32, O.BF16))
