"""MaxPool2d on the K x K window kernel and the LDS tile backward, bit-exact
against the numpy restatement at the sizes where they can go wrong: planes that
share workgroups with a ragged last one, rows of 4 and not of 4 elements,
planes past the LDS tile, padding in every mode, ties, infinities and NaN, and
views that start between 16-byte boundaries."""
import numpy as np
import pytest
import torch

from novann_amd import functional as F
from oracle import functional_ref as R

pytestmark = pytest.mark.gpu

# (N, C, H, W, k, s, p)
SHAPES = [
    (1, 1, 1, 1, 2, 1, 1), (1, 3, 2, 3, 2, 2, 0), (3, 7, 7, 7, 3, 2, 1), (130, 33, 7, 7, 3, 2, 1),
    (2, 9, 28, 28, 3, 2, 1), (2, 5, 12, 16, 3, 1, 1), (3, 4, 9, 9, 3, 3, 0), (2, 3, 15, 15, 2, 2, 0),
    (5, 3, 11, 8, 3, 1, 2), (2, 3, 13, 20, 5, 3, 2), (1, 2, 120, 120, 3, 2, 1), (2, 2, 6, 40, 2, 3, 1),
    (9, 64, 8, 8, 2, 2, 0),
]


def values(rng, shape, special):
    x = np.round(rng.standard_normal(shape) * 2).astype(np.float32) / 2  # many ties, both zeros
    x[rng.random(shape) < 0.1] = -0.0
    if special:
        flat = x.reshape(-1)
        for v in (np.inf, -np.inf, np.nan, -np.inf):
            flat[rng.integers(0, flat.size)] = v
        x[..., :1, :] = -np.inf
    return x


@pytest.mark.parametrize("mode", ["zeros", "reflect", "replicate", "circular"])
@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_windows_bit_exact(shape, special, mode):
    n, c, h, w, k, s, p = shape
    if mode != "zeros" and (p == 0 or p >= min(h, w)):
        pytest.skip("no padding to resolve")
    print(f"pool {shape} {mode} special {special}", flush=True)
    rng = np.random.default_rng(sum(shape))
    x = values(rng, (n, c, h, w), special)
    y = R.max_pool2d(x, (k, k), (s, s), (p, p), mode)
    g = rng.standard_normal(y.shape).astype(np.float32)
    if special:
        g.reshape(-1)[rng.integers(0, g.size)] = np.inf
    with np.errstate(invalid="ignore"):
        gi = R.max_pool2d_backward(g, x, (k, k), (s, s), (p, p), mode)
    # views 4 bytes past a 16-byte boundary too
    for shift in (0, 1):
        def put(a):
            t = torch.empty(a.size + shift, dtype=torch.float32, device="cuda")[shift:]
            t.copy_(torch.from_numpy(a.reshape(-1)))
            return t.view(a.shape)
        xd, gd = put(x), put(g)
        got = F.max_pool2d(xd, k, s, p, mode).cpu().numpy()
        assert np.array_equal(got.view(np.uint32), y.view(np.uint32)) or (
            np.array_equal(np.isnan(got), np.isnan(y))
            and np.array_equal(got[~np.isnan(y)].view(np.uint32), y[~np.isnan(y)].view(np.uint32)))
        got = F.max_pool2d_backward(gd, xd, k, s, p, mode).cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(gi))
        assert np.array_equal(got[~np.isnan(gi)].view(np.uint32), gi[~np.isnan(gi)].view(np.uint32))


# few large planes: walked an element a lane; one pixel or plane less in tiles
FEW = [(1, 3, 57, 58, 2, 2, 0), (1, 64, 57, 58, 3, 3, 0), (2, 2, 90, 91, 2, 3, 0),
       (1, 2, 45, 45, 2, 2, 0), (1, 4, 80, 80, 3, 2, 1), (17, 1, 80, 80, 3, 2, 1)]


@pytest.mark.parametrize("shape", FEW, ids=lambda s: "x".join(map(str, s)))
def test_few_large_planes_bit_exact(shape):
    for special in (False, True):
        test_windows_bit_exact(shape, special, "zeros")
