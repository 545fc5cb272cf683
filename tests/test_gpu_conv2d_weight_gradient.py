"""grad_weight and grad_bias of stride-1 convolutions at the sizes where their
kernels can go wrong: rows staged in runs of 2 (even widths that are no
multiple of 4, on either side), bands that do not divide the output rows,
channel blocks that are not whole, and column sums of four columns a lane whose
last workgroup is not whole, over one and several partials.

The bar is derived: grad and x enter the products rounded to bf16, so only the
fp32 sums differ from fp64, by at most (n + 1) * 2^-23 times the sum of
|products| for n products; grad_bias adds the unrounded values."""
import numpy as np
import pytest
import torch

from novann_amd import functional as F
from novann_amd.module import QuantizedParameters
from tests.gpu_util import bf16_round

pytestmark = pytest.mark.gpu

# (N, C, H, W, C_out, k, padding)
SHAPES = [
    (3, 16, 14, 14, 20, 3, 1),     # two bands, the second short
    (2, 33, 9, 30, 65, 3, 1),      # 32-pixel rows, channel blocks and one more
    (5, 16, 7, 16, 17, 3, 0),      # W a multiple of 4, OW not
    (2, 20, 6, 14, 16, 3, 2),      # OW a multiple of 4, W not
    (1, 17, 5, 2, 16, 3, 1),       # two pixels a row
    (1, 32, 12, 46, 40, 3, 1),     # 64-pixel rows
    (1, 76, 6, 6, 100, 3, 1),      # 68400 columns: 267 workgroups and a rest, one partial
    (40, 68, 5, 10, 116, 3, 1),    # 70992 columns, several partials
    (9, 260, 4, 4, 256, 1, 0),     # 66560 columns of a 1 x 1 window
]


def col(x, k, p):
    """(N, C, k, k, OH, OW) windows of the zero-padded input, float64."""
    xp = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (p, p), (p, p)))
    return np.lib.stride_tricks.sliding_window_view(xp, (k, k), (2, 3)).transpose(0, 1, 4, 5, 2, 3)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_weight_and_bias_gradients(shape):
    print(f"weight gradient {shape}", flush=True)
    n, c, h, w, co, k, p = shape
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    g = rng.standard_normal((n, co, h + 2 * p - k + 1, w + 2 * p - k + 1)).astype(np.float32)
    q = QuantizedParameters.from_float(rng.standard_normal((co, c, k, k)).astype(np.float32), "e4m3")
    xd, gd = torch.from_numpy(x).cuda(), torch.from_numpy(g).cuda()
    _, gw, gb = F.conv2d_backward(gd, xd, q, k, 1, p)
    xb, gr = bf16_round(x), bf16_round(g).astype(np.float64)
    want = np.tensordot(gr, col(xb, k, p), ((0, 2, 3), (0, 4, 5)))
    mag = np.tensordot(np.abs(gr), col(np.abs(xb), k, p), ((0, 2, 3), (0, 4, 5)))
    terms = g[:, 0].size
    assert np.all(np.abs(gw.cpu().numpy() - want) <= (terms + 1) * 2.0**-23 * mag + 1e-30)
    want_b, mag_b = (f(g.astype(np.float64)).sum(axis=(0, 2, 3)) for f in (np.asarray, np.abs))
    assert np.all(np.abs(gb.cpu().numpy()[:, 0] - want_b) <= (terms + 1) * 2.0**-23 * mag_b)
    # the sums run in a fixed order
    _, gw2, gb2 = F.conv2d_backward(gd, xd, q, k, 1, p)
    assert torch.equal(gw, gw2) and torch.equal(gb, gb2)
