"""Linear products whose rows are read by quads of lanes, 128 elements a block:
first and last block counts a wave takes, every kind of rest (none, below and
above 64, odd), rows and features short of a tile and of a quad's 4 rows, every
stored type, and non-finite values just outside what a product reads.

The bar is derived as for the other split products: the operands are known
exactly, so only the fp32 sums differ from fp64, by at most K * 2^-23 times the
sum of |products|."""
import numpy as np
import pytest
import torch

from novann_amd import functional as F
from novann_amd import quant
from tests.gpu_util import bf16_round
from tests.test_gpu_linear_split import check, weight

pytestmark = pytest.mark.gpu

# (rows, D_in, D_out)
SHAPES = [(4, 2048, 1), (5, 2049, 15), (16, 2111, 17), (7, 4224, 33),   # 16 x 16 tiles
          (17, 512, 3), (31, 575, 33), (33, 576, 30), (63, 639, 65),    # 32 x 32 tiles
          (18, 1151, 31), (520, 1024, 530), (300, 2050, 1030)]


@pytest.mark.parametrize("wdt", ["e4m3", "e5m2", "e2m1"])
@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16, torch.float16])
def test_quad_rows_exact_operands(m, k, n, wdt, xdt):
    print(f"quad forward {wdt} {xdt} {m}x{k}x{n}", flush=True)
    rng = np.random.default_rng(m * 31 + k * 7 + n)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).cuda().to(xdt)
    q, w = weight(rng, n, k, wdt)
    y = F.linear(x, q).cpu().numpy()
    check(y, bf16_round(x.float().cpu().numpy()).astype(np.float64), w.T.astype(np.float64),
          (m, k, n, wdt))


@pytest.mark.parametrize("m,k,n", [SHAPES[1], SHAPES[5]])
def test_quad_rows_fp8_input(m, k, n):
    rng = np.random.default_rng(k)
    xq = quant.quantize(torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).cuda(),
                        "e5m2")
    q, w = weight(rng, n, k, "e4m3")
    y = F.linear(xq, q).cpu().numpy().astype(np.float64)
    x = quant.dequantize(xq).cpu().numpy().astype(np.float64)
    # the scales are applied after the sums: one more rounding
    bound = (k + 2) * 2.0**-23 * (np.abs(x) @ np.abs(w.T)) + 1e-30
    assert np.all(np.abs(y - x @ w.T) <= bound)


@pytest.mark.parametrize("m,k,n", [(5, 2049, 15), (33, 639, 31)])
def test_quad_rows_read_nothing_past_the_operands(m, k, n):
    """Rows of a larger NaN-filled buffer: a row's rest and the tile's missing
    rows come from inside x."""
    rng = np.random.default_rng(m)
    buf = torch.full((m * k + 4096,), float("nan"), device="cuda")
    x = rng.standard_normal((m, k)).astype(np.float32)
    buf[:m * k] = torch.from_numpy(x).cuda().reshape(-1)
    q, w = weight(rng, n, k, "e4m3")
    y = F.linear(buf[:m * k].view(m, k), q).cpu().numpy()
    check(y, bf16_round(x).astype(np.float64), w.T.astype(np.float64), (m, k, n))


def test_quad_rows_keep_nan_in_its_row():
    rng = np.random.default_rng(1)
    x = rng.standard_normal((40, 1024)).astype(np.float32)
    x[21, 700] = np.nan
    q, _ = weight(rng, 48, 1024, "e4m3")
    y = F.linear(torch.from_numpy(x).cuda(), q).cpu().numpy()
    bad = np.isnan(y)
    assert bad[21].all() and bad.sum() == 48
