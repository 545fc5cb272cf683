"""Linear products on the split-K kernel and on the 128 x 256-tile kernels'
ragged forms, at the sizes where they can go wrong: one element past and short
of a tile, a K block, a wave's share of K; and non-finite values just outside
what a product reads.

The bar is derived: the operands the MFMAs multiply are known exactly (x and
grad rounded to bf16, W's codes), so only the fp32 sums differ from fp64, by at
most K * 2^-23 times the sum of |products| (each addition rounds once, the MFMA
may round both of its internal steps)."""
import numpy as np
import pytest
import torch

import oracle as O
from novann_amd import functional as F
from novann_amd.module import Parameters, QuantizedParameters
from tests.gpu_util import bf16_round

pytestmark = pytest.mark.gpu


def check(got, x, w, what):
    """got against x @ w (both float64, the exact operands)."""
    bound = max(x.shape[1], 8) * 2.0**-23 * (np.abs(x) @ np.abs(w)) + 1e-30
    assert np.all(np.abs(got.astype(np.float64) - x @ w) <= bound), what


def weight(rng, n, k, wdt):
    w = (rng.standard_normal((n, k)) * 0.1).astype(np.float32)
    if wdt in ("f32", "bf16"):
        t = torch.from_numpy(w).cuda()
        return Parameters(t if wdt == "f32" else torch.from_numpy(bf16_round(w)).cuda()), bf16_round(w)
    q = QuantizedParameters.from_float(w, wdt)
    return q, q.dequantize().cpu().numpy()


# (rows, D_in, D_out): the 16 x 16, 32 x 32 and 64 x 64 tiles of the split
# kernel, its K blocks of 64 over 16, 8 and 4 waves, odd rows in every format
SPLIT = [(1, 1, 1), (1, 64, 16), (3, 1030, 17), (16, 1025, 15), (17, 63, 33), (33, 129, 31),
         (64, 577, 65), (129, 640, 40), (1025, 65, 1030), (1030, 333, 1025)]


@pytest.mark.parametrize("wdt", ["e4m3", "e2m1", "f32"])
@pytest.mark.parametrize("m,k,n", SPLIT)
@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16, torch.float16])
def test_split_forward_exact_operands(m, k, n, wdt, xdt):
    print(f"split forward {wdt} {xdt} {m}x{k}x{n}", flush=True)
    rng = np.random.default_rng(m * 31 + k * 7 + n)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).cuda().to(xdt)
    q, w = weight(rng, n, k, wdt)
    y = F.linear(x, q).cpu().numpy()
    check(y, bf16_round(x.float().cpu().numpy()).astype(np.float64), w.T.astype(np.float64),
          (m, k, n, wdt))


# (N, D_in, D_out): grad_input and grad_weight on the split kernel (at least 4
# features each way), one feature less than that, and the ragged tile kernels
# (more than 32 tiles of 128 x 256)
BACKWARD = [(1, 4, 4), (3, 5, 7), (65, 4, 70), (64, 66, 4), (129, 33, 65), (257, 100, 36),
            (70, 3, 40), (70, 40, 2), (1030, 1040, 1004), (130, 2052, 1160)]


@pytest.mark.parametrize("wdt", ["e4m3", "e2m1", "f32"])
@pytest.mark.parametrize("n,d_in,d_out", BACKWARD)
def test_backward_exact_operands(n, d_in, d_out, wdt):
    print(f"linear backward {wdt} {n}x{d_in}x{d_out}", flush=True)
    rng = np.random.default_rng(n * 31 + d_in * 7 + d_out)
    x = rng.standard_normal((n, d_in)).astype(np.float32)
    g = rng.standard_normal((n, d_out)).astype(np.float32)
    q, w = weight(rng, d_out, d_in, wdt)
    gi, gw, gb = F.linear_backward(torch.from_numpy(g).cuda(), torch.from_numpy(x).cuda(), q)
    g16, x16 = bf16_round(g).astype(np.float64), bf16_round(x).astype(np.float64)
    check(gi.cpu().numpy(), g16, w.astype(np.float64), "grad_input")
    check(gw.cpu().numpy(), g16.T, x16, "grad_weight")
    check(gb.cpu().numpy().reshape(1, -1), np.ones((1, n)), g.astype(np.float64), "grad_bias")


# One to T - 1 indices of W's columns (D_in), of x's and of grad's left for the
# last tile of T-wide runs: T = 2 (32 x 32 tiles), 4 (64 x 64) and both (64 x 32).
EDGES = [(5, 33, 97), (40, 65, 33), (1024, 1025, 44), (1023, 1026, 36), (1025, 1027, 20),
         (20, 1024, 1025), (12, 1025, 1026), (9, 1057, 1027)]


@pytest.mark.parametrize("wdt", ["e4m3", "e2m1", "f32"])
@pytest.mark.parametrize("n,d_in,d_out", EDGES)
def test_backward_of_a_few_indices_past_a_tile(n, d_in, d_out, wdt):
    test_backward_exact_operands(n, d_in, d_out, wdt)


# more than 32 tiles of 128 x 256, ragged in M, N and K
RAGGED = [(1026, 144, 1003), (1100, 32, 1280), (1024, 416, 1025), (4100, 160, 250)]


@pytest.mark.parametrize("wdt", ["e4m3", "e5m2", "e2m1"])
@pytest.mark.parametrize("m,k,n", RAGGED)
@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16])
def test_ragged_tiles_read_nothing_outside(m, k, n, wdt, xdt):
    """Row 7 of W and of x hold NaN (for E2M1, which has none, row 7 of x
    only): exactly that output column and that output row are NaN, so no
    neighbouring row's values enter where K ends inside a block."""
    print(f"ragged {wdt} {xdt} {m}x{k}x{n}", flush=True)
    rng = np.random.default_rng(m + k + n)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).cuda()
    x[7] = float("nan")
    x = x.to(xdt)
    q, w = weight(rng, n, k, wdt)
    if wdt != "e2m1":
        q.codes.view(torch.uint8).view(n, k)[7] = 0x7F
    y = F.linear(x, q).cpu().numpy()
    nan = np.zeros((m, n), bool)
    nan[7] = True
    if wdt != "e2m1":
        nan[:, 7] = True
    assert np.array_equal(np.isnan(y), nan)
    rows, cols = [i for i in range(m) if i != 7], [j for j in range(n) if j != 7 or wdt == "e2m1"]
    check(y[rows][:, cols], bf16_round(x.float().cpu().numpy()[rows]).astype(np.float64),
          w[cols].T.astype(np.float64), (m, k, n))


def test_ragged_grad_input_reads_nothing_outside():
    """grad_input on W's codes in place, the batch and both features ragged:
    a NaN column of W makes one NaN column, a NaN row of grad one NaN row."""
    n, d_in, d_out = 1030, 1040, 1000
    rng = np.random.default_rng(5)
    g = rng.standard_normal((n, d_out)).astype(np.float32)
    g[9] = np.nan
    q, w = weight(rng, d_out, d_in, "e4m3")
    q.codes.view(torch.uint8).view(d_out, d_in)[:, 5] = 0x7F
    gi, _, _ = F.linear_backward(torch.from_numpy(g).cuda(),
                                 torch.zeros((n, d_in), device="cuda"), q)
    gi = gi.cpu().numpy()
    nan = np.zeros((n, d_in), bool)
    nan[9] = nan[:, 5] = True
    assert np.array_equal(np.isnan(gi), nan)
    rows, cols = [i for i in range(n) if i != 9], [j for j in range(d_in) if j != 5]
    check(gi[rows][:, cols], bf16_round(g[rows]).astype(np.float64),
          w[:, cols].astype(np.float64), "grad_input")


@pytest.mark.parametrize("m,k,n", [(5, 70, 37), (70, 131, 130), (1026, 144, 1003)])
def test_epilogue_on_ragged_shapes(m, k, n):
    """The fused epilogue equals its steps on the plain output bit for bit, and
    the amax covers what is stored and nothing else."""
    rng = np.random.default_rng(m)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).cuda()
    q, _ = weight(rng, n, k, "e4m3")
    mul = rng.standard_normal(n).astype(np.float32)
    add = rng.standard_normal(n).astype(np.float32)
    amax = torch.zeros(1, device="cuda")
    y = F.linear(x, q).cpu().numpy()
    got = F.linear(x, q, epilogue=F.Epilogue(channel_mul=mul, channel_add=add, relu=True,
                                             out_dtype="bf16", out_amax=amax))
    v = y * mul + add
    v = v * (v > 0)
    want = O.cast(v.reshape(-1).astype(np.float32), O.F32, O.BF16)
    assert np.array_equal(got.view(torch.int16).cpu().numpy().view(np.uint16).reshape(-1), want)
    assert float(amax) == np.abs(v).max()
