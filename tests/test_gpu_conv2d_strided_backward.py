"""The input gradient of strided and widely padded convolutions (fp32 sums, one
residue class of pixels a workgroup) at the sizes where it can go wrong:
strides above the window and above the image, channel blocks and stages of 128
output channels that are not whole, one pixel past a workgroup, both ways of
splitting the work; and a NaN weight, which reaches the pixels its tap reaches
and no others.

The bar is derived: grad and the decoded weights are exact, so only fp32
roundings differ from fp64, at most (K + 2) * 2^-24 times the sum of |products|
with K = C_out * KH * KW."""
import numpy as np
import pytest
import torch

from novann_amd import _lib
from novann_amd import functional as F
from novann_amd.module import Parameters, QuantizedParameters
from oracle import functional_ref as R

pytestmark = pytest.mark.gpu

# (N, C, H, W, C_out, KH, KW, stride, pad)
SHAPES = [
    (1, 1, 5, 4, 1, 3, 3, (2, 2), (1, 1)),
    (3, 9, 13, 11, 129, 3, 3, (2, 2), (1, 1)),     # one channel past a stage
    (2, 17, 9, 10, 128, 1, 1, (2, 2), (0, 0)),     # taps of one phase in four
    (2, 16, 8, 7, 5, 2, 3, (5, 4), (0, 1)),        # strides above the window
    (2, 4, 3, 3, 6, 3, 3, (7, 9), (2, 2)),         # and above the image
    (5, 33, 14, 14, 20, 5, 5, (2, 3), (2, 4)),
    (1, 3, 6, 6, 7, 3, 3, (1, 1), (4, 3)),         # stride 1, padding past the window
    (65, 8, 4, 4, 130, 3, 3, (2, 2), (1, 1)),      # 260 pixels a phase
    (70, 130, 18, 18, 32, 3, 3, (2, 2), (1, 1)),   # many workgroups of 256 pixels
    # the taps' phases alone: one pixel each and a few, taps on the padding, pixels
    # past the image
    (3, 20, 70, 80, 6, 2, 3, (70, 80), (0, 0)),
    (1, 3, 131, 127, 5, 3, 2, (90, 100), (1, 0)),
    (2, 130, 33, 34, 7, 3, 3, (40, 32), (2, 7)),
]


def gradients(x, q, g, case):
    gi, _, _ = F.conv2d_backward(torch.from_numpy(g).cuda(), torch.from_numpy(x).cuda(), q,
                                 (case[5], case[6]), case[7], case[8])
    return gi.cpu().numpy()


@pytest.mark.parametrize("wdt", ["e4m3", "e2m1", "f32"])
@pytest.mark.parametrize("case", SHAPES, ids=lambda c: "x".join(map(str, c[:7])))
def test_strided_grad_input(case, wdt):
    n, c, h, w, co, kh, kw, st, pad = case
    print(f"strided backward {case} {wdt}", flush=True)
    rng = np.random.default_rng(n + c + h + co)
    x = np.zeros((n, c, h, w), np.float32)
    wt = (rng.standard_normal((co, c, kh, kw)) * 0.1).astype(np.float32)
    if wdt == "f32":
        q, wd = Parameters(torch.from_numpy(wt).cuda()), wt
    else:
        q = QuantizedParameters.from_float(wt, wdt)
        wd = q.dequantize().cpu().numpy()
    oh, ow = (h + 2 * pad[0] - kh) // st[0] + 1, (w + 2 * pad[1] - kw) // st[1] + 1
    g = rng.standard_normal((n, co, oh, ow)).astype(np.float32)
    got = gradients(x, q, g, case)
    x64, w64, g64 = x.astype(np.float64), wd.astype(np.float64), g.astype(np.float64)
    want = R.conv2d_backward(g64, x64, w64, st, pad)[0]
    size = R.conv2d_backward(np.abs(g64), x64, np.abs(w64), st, pad)[0]
    assert np.all(np.abs(got - want) <= (co * kh * kw + 2) * 2.0**-24 * size + 1e-30), case


def test_nan_weight_reaches_only_its_taps_pixels():
    case = (2, 16, 8, 8, 24, 3, 3, (2, 2), (1, 1))
    rng = np.random.default_rng(1)
    x = np.zeros(case[:4], np.float32)
    q = QuantizedParameters.from_float((rng.standard_normal((24, 16, 3, 3)) * 0.1).astype(np.float32),
                                       "e4m3")
    g = rng.standard_normal((2, 24, 4, 4)).astype(np.float32)
    clean = gradients(x, q, g, case)
    q.codes.view(torch.uint8).view(24, 16, 3, 3)[3, 5, 0, 0] = 0x7F
    got = gradients(x, q, g, case)
    hit = np.zeros(case[:4], bool)
    hit[:, 5, 1:7:2, 1:7:2] = True  # pixels 2 oh - 1 of tap (0, 0), oh = 1, 2, 3
    assert np.array_equal(np.isnan(got), hit)
    assert np.array_equal(got[~hit], clean[~hit])


@pytest.mark.parametrize("stride", [(2**31 - 1, 2**31 - 1), (2**31 - 1, 2), (3, 2**31 - 3)])
def test_strides_up_to_the_largest_int(stride):
    """One output row (column): only the first window's pixels get a gradient,
    every other pixel is zero, and no tap past the window is looked for."""
    n, c, h, w, co, k, pad = 2, 17, 6, 9, 5, 3, (1, 1)
    rng = np.random.default_rng(2)
    wt = (rng.standard_normal((co, c, k, k)) * 0.1).astype(np.float32)
    q = QuantizedParameters.from_float(wt, "e4m3")
    oh, ow = ((d + 2 * p - k) // s + 1 for d, p, s in zip((h, w), pad, stride))
    g = rng.standard_normal((n, co, oh, ow)).astype(np.float32)
    gi = torch.full((n, c, h, w), float("nan"), device="cuda")
    lib, gd = _lib.load(), torch.from_numpy(g).cuda()
    code = _lib.DTYPES["e4m3"]
    work = torch.empty(lib.novaq_conv2d_backward_workspace(n, c, co, k, k, code) + 16,
                       dtype=torch.uint8, device="cuda")
    # grad_input alone
    _lib.check(lib.novaq_conv2d_backward(
        gd.data_ptr(), None, n, c, h, w, q.codes.data_ptr(), code, q.scale.data_ptr(), co, k, k,
        *stride, *pad, 0, gi.data_ptr(), None, None, work.data_ptr(), work.numel(),
        torch.cuda.current_stream().cuda_stream), "conv2d backward")
    # the same windows at a stride that fits the padded image
    near = tuple(min(s, d + 2 * p) for s, d, p in zip(stride, (h, w), pad))
    w64 = q.dequantize().cpu().numpy().astype(np.float64)
    x64, g64 = np.zeros((n, c, h, w)), g.astype(np.float64)
    want = R.conv2d_backward(g64, x64, w64, near, pad)[0]
    size = R.conv2d_backward(np.abs(g64), x64, np.abs(w64), near, pad)[0]
    got = gi.cpu().numpy()
    assert np.all(np.abs(got - want) <= (co * k * k + 2) * 2.0**-24 * size + 1e-30)
    assert not got[size == 0].any()
