"""Linear products on the kernels of 128-row tiles, which run where 128 x 256
tiles cover more than an eighth of the CUs: the ping-pong kernel (FP8 W), the
wide-K kernel (FP4 W), their ragged forms, and the staged-decode kernel (16-bit
W, and whole tiles that the other two do not have); and the backward's
weight-gradient kernel of such tiles with the bf16 copy of grad that it leaves.

The bar is derived: the operands the MFMAs multiply are known exactly, so only
the fp32 sums differ from fp64, by at most K * 2^-23 times the sum of
|products|, and the scale, applied after them, adds a rounding."""
import numpy as np
import pytest
import torch

import oracle as O
from novann_amd import _lib
from novann_amd import functional as F
from tests.gpu_util import bf16_round
from tests.test_gpu_epilogue import (check_all_outputs, combined_scale, linear_ex, linear_x,
                                     quantized_codes, x_codes)
from tests.test_gpu_linear import QCODE, dequant, run_linear, valid_codes
from tests.test_gpu_linear_split import check, weight

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


# wdt, M, K, N: each kernel with at least one tile past an eighth of the CUs
KERNELS = [
    ("e4m3", 1024, 256, 2304),   # ping-pong
    ("e5m2", 4224, 128, 256),    # ping-pong, one K block
    ("e2m1", 1024, 384, 2304),   # wide-K
    ("e4m3", 1026, 144, 1003),   # ping-pong, ragged
    ("e2m1", 1100, 96, 1290),    # wide-K, ragged
    ("e2m1", 1152, 64, 1280),    # staged-decode, 256 columns
    ("e4m3", 2048, 192, 640),    # staged-decode, 128 columns
    ("bf16", 1152, 128, 1280),   # staged-decode, 16-bit weights
    ("f16", 2048, 64, 640),
]


@pytest.mark.parametrize("wdt,m,k,n", KERNELS)
def test_epilogue_bit_exact(wdt, m, k, n):
    """The fused affine, ReLU, amax and every narrow store equal the oracle's
    steps on the plain output bit for bit; the plain output is exact to its
    sums."""
    print(f"tile epilogue {wdt} {m}x{k}x{n}", flush=True)
    assert takes_tiles(m, n)
    rng = np.random.default_rng(m + k + n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    w = (rng.standard_normal((n, k)) * 0.1).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    wd, ws, wdeq = quantized_codes(w, wdt, rng)
    y0 = linear_ex(x, wd, wdt, ws, n, None, bias)
    a = bf16_round(x).astype(np.float64)
    b = (wdeq if ws is not None else bf16_round(wdeq)).astype(np.float64).T
    bound = (k + 2) * 2.0**-23 * (np.abs(a) @ np.abs(b) + np.abs(bias)) + 1e-30
    assert np.all(np.abs(y0.view(np.float32) - (a @ b + bias)) <= bound)
    check_all_outputs(lambda ep: linear_ex(x, wd, wdt, ws, n, ep, bias), y0, n, rng)


@pytest.mark.parametrize("xt", ["bf16", "f16", "e4m3", "e5m2"])
@pytest.mark.parametrize("wdt,m,k,n", [KERNELS[0], KERNELS[3], KERNELS[4], KERNELS[5],
                                       KERNELS[6], KERNELS[7]])
def test_stored_activations(xt, wdt, m, k, n):
    """x stored as xt gives the fp32-input product on the decoded x with the
    scale folded into the weights': bit for bit where the kernel is the same,
    else (FP8 x and W: other kernels) to the sums' roundings."""
    rng = np.random.default_rng(m * 3 + k + n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    w = (rng.standard_normal((n, k)) * 0.1).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    wd, ws, wdeq = quantized_codes(w, wdt, rng)
    xd, sx, xdec = x_codes(x, xt)
    got = linear_x(xd, xt, sx, m, k, wd, wdt, ws, n, bias).view(np.float32)
    want = linear_x(torch.from_numpy(np.ascontiguousarray(xdec)).cuda(), "f32", None, m, k, wd,
                    wdt, combined_scale(ws, sx), n, bias).view(np.float32)
    if xt in ("bf16", "f16") or wdt == "bf16":
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    else:
        size = np.abs(xdec.astype(np.float64)) @ np.abs(wdeq.astype(np.float64)).T * float(sx)
        bound = 2 * (k + 3) * 2.0**-23 * (size + np.abs(bias)) + 1e-30
        assert np.all(np.abs(got.astype(np.float64) - want) <= bound)


@pytest.mark.parametrize("wdt", ["e4m3", "e5m2", "e2m1"])
@pytest.mark.parametrize("m,k,n", [(1024, 256, 2304), (1152, 192, 1280), (2048, 128, 640),
                                   (1030, 224, 1290)],
                         ids=["whole", "staged-256", "staged-128", "ragged"])
def test_identity_input_reproduces_dequantized_weights_exactly(wdt, m, k, n):
    """x = I: y[i, j] = s * dec(W[j, i]) exactly, for every finite code, on each
    kernel's decode and lane layout."""
    assert takes_tiles(m, n)
    rng = np.random.default_rng(1)
    vals = valid_codes(wdt)
    nib = vals[rng.integers(0, vals.size, size=n * k)]
    nib[: vals.size] = vals
    codes = (nib[0::2] | (nib[1::2] << 4)).astype(np.uint8) if wdt == "e2m1" else nib.astype(np.uint8)
    x = np.zeros((m, k), np.float32)
    x[:k] = np.eye(k, dtype=np.float32)
    y = run_linear(x, codes, wdt, 0.0123, None, n, k)
    w = dequant(codes, wdt, n * k, 0.0123).reshape(n, k)
    assert np.array_equal(y[:k], np.ascontiguousarray(w.T))
    assert not np.any(y[k:])


@pytest.mark.parametrize("wdt", ["e4m3", "e2m1"])
def test_longest_k_one_hot_rows(wdt):
    """K = 2^21, the longest the K-block kernels take, on 33 tiles: one-hot rows
    of x (of grad) pick columns of W spread over the whole of K, so y (and
    grad_input, W's FP8 codes read in their [K][N] layout) is exact -- the
    offsets of the last K blocks, near the top of the 31-bit buffer ranges."""
    M, N, K = 4224, 256, 1 << 21
    assert takes_tiles(M, N)
    print(f"longest K one-hot tiles {wdt}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(21)
    stored = K // 2 if wdt == "e2m1" else K
    codes = torch.randint(0, 256, (N, stored), generator=g, device="cuda", dtype=torch.uint8)
    if wdt == "e4m3":  # no NaN codes
        codes -= ((codes & 0x7F) == 0x7F).to(torch.uint8)
    s = 0.0123
    sd = torch.tensor([s], dtype=torch.float32, device="cuda")
    rng = np.random.default_rng(21)
    ks = rng.integers(0, K, size=M)
    ks[0], ks[1], ks[2], ks[-1] = 0, K - 1, K - 128, K - 2
    kd = torch.from_numpy(ks).cuda()
    rows = torch.arange(M, device="cuda")
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    code = _lib.DTYPES[wdt]
    x = torch.zeros((M, K), dtype=torch.float32, device="cuda")
    x[rows, kd] = 1.0
    y = torch.empty((M, N), dtype=torch.float32, device="cuda")
    _lib.check(lib.novaq_linear_forward(x.data_ptr(), M, K, codes.data_ptr(), code, sd.data_ptr(),
                                        None, N, y.data_ptr(), stream), "linear")
    picked = codes[:, kd // 2 if wdt == "e2m1" else kd].t().contiguous().cpu().numpy()
    if wdt == "e2m1":
        picked = np.where((ks % 2 == 1)[:, None], picked >> 4, picked & 0xF).astype(np.uint8)
        flat = picked.reshape(-1)
        want = O.cast((flat[0::2] | (flat[1::2] << 4)).astype(np.uint8), O.E2M1, O.F32, n=flat.size,
                      scale=s)
    else:
        want = O.cast(picked.reshape(-1), QCODE[wdt], O.F32, scale=s)
    # (a -0 weight sums to +0 with the other products' zeros)
    assert np.array_equal(y.cpu().numpy(), want.view(np.float32).reshape(M, N))
    if wdt == "e2m1":
        return
    # W (D_out = K, D_in = N): the same bytes read as [K][N], x as grad
    y.fill_(float("nan"))
    work = torch.empty(lib.novaq_linear_backward_workspace(M, N, K, code), dtype=torch.uint8,
                       device="cuda")
    _lib.check(lib.novaq_linear_backward(
        x.data_ptr(), None, M, N, codes.data_ptr(), code, sd.data_ptr(), K, y.data_ptr(), None,
        None, work.data_ptr(), work.numel(), stream), "linear backward")
    picked = codes.view(K, N)[kd].contiguous().cpu().numpy()
    want = O.cast(picked.reshape(-1), QCODE[wdt], O.F32, scale=s).view(np.float32).reshape(M, N)
    assert np.array_equal(y.cpu().numpy(), want)


# (N, D_in, D_out) with E2M1 weights, whose grad_input multiplies the bf16 grad
# that the weight-gradient kernel stores: its 128 x 256 and 256 x 256 tiles, whole
# and ragged
@pytest.mark.parametrize("n,d_in,d_out", [(1024, 2048, 1152), (1030, 2052, 1184),
                                          (384, 4096, 4096), (390, 4100, 4096)])
def test_weight_gradient_tiles_leave_grad_in_bf16(n, d_in, d_out):
    print(f"tile backward e2m1 {n}x{d_in}x{d_out}", flush=True)
    assert takes_tiles(n, d_in) and takes_tiles(d_out, d_in) and d_out % 32 == 0
    rng = np.random.default_rng(n + d_in)
    x = rng.standard_normal((n, d_in)).astype(np.float32)
    g = rng.standard_normal((n, d_out)).astype(np.float32)
    q, w = weight(rng, d_out, d_in, "e2m1")
    gi, gw, gb = F.linear_backward(torch.from_numpy(g).cuda(), torch.from_numpy(x).cuda(), q)
    g16, x16 = bf16_round(g).astype(np.float64), bf16_round(x).astype(np.float64)
    check(gi.cpu().numpy(), g16, w.astype(np.float64), "grad_input")
    check(gw.cpu().numpy(), g16.T, x16, "grad_weight")
    check(gb.cpu().numpy().reshape(1, -1), np.ones((1, n)), g.astype(np.float64), "grad_bias")
