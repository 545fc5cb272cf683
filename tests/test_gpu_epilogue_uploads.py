"""Host-array channel vectors of a fused epilogue are copied without waiting
for the GPU: every call has to see its own values, also while earlier calls are
still queued, on several streams, and whichever of the two vectors is given."""
import numpy as np
import pytest
import torch

from novann_amd import functional as F
from novann_amd.module import QuantizedParameters

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D_out", [1, 5, 64, 1027])
def test_queued_calls_see_their_own_vectors(D_out):
    rng = np.random.default_rng(D_out)
    x = torch.from_numpy(rng.standard_normal((8, 64)).astype(np.float32)).cuda()
    q = QuantizedParameters.from_float(rng.standard_normal((D_out, 64)).astype(np.float32), "e4m3")
    y = F.linear(x, q)
    big = torch.empty(1 << 26, device="cuda")
    streams = [torch.cuda.current_stream(), torch.cuda.Stream()]
    streams[1].wait_stream(streams[0])
    runs = []
    for i in range(40):
        # float64 and strided arrays round and flatten as numpy does
        mul = rng.standard_normal((D_out, 2))[:, 0]
        add = rng.standard_normal(D_out).astype(np.float32) if i % 3 else None
        with torch.cuda.stream(streams[i % 2]):
            if i % 10 == 0:
                big.fill_(i)  # keeps the queue busy while the next calls are made
            got = F.linear(x, q, epilogue=F.Epilogue(channel_mul=mul, channel_add=add))
        runs.append((got, mul.astype(np.float32), add))
        mul[:] = np.nan  # the caller's array is free after the call
    torch.cuda.synchronize()
    yh = y.cpu().numpy()
    for got, mul, add in runs:
        want = yh * mul if add is None else yh * mul + add
        assert np.array_equal(got.cpu().numpy(), want)


def test_device_and_host_vectors_mix_and_sizes_are_checked():
    rng = np.random.default_rng(0)
    x = torch.from_numpy(rng.standard_normal((4, 32)).astype(np.float32)).cuda()
    q = QuantizedParameters.from_float(rng.standard_normal((6, 32)).astype(np.float32), "e4m3")
    mul = rng.standard_normal(6).astype(np.float32)
    add = torch.from_numpy(rng.standard_normal(6).astype(np.float32)).cuda()
    y = F.linear(x, q).cpu().numpy()
    got = F.linear(x, q, epilogue=F.Epilogue(channel_mul=mul, channel_add=add)).cpu().numpy()
    assert np.array_equal(got, y * mul + add.cpu().numpy())
    for bad in (dict(channel_mul=mul[:5]), dict(channel_mul=mul, channel_add=np.ones(7))):
        with pytest.raises(ValueError, match="values, expected 6"):
            F.linear(x, q, epilogue=F.Epilogue(**bad))
    with pytest.raises(TypeError):
        F.linear(x, q, epilogue=F.Epilogue(channel_mul=[1.0] * 6))


def test_layer_without_outputs_takes_empty_vectors():
    x = torch.zeros((3, 8), device="cuda")
    w = torch.zeros((0, 8), device="cuda")
    none = np.zeros(0, np.float32)
    for kw in (dict(channel_mul=none), dict(channel_add=none),
               dict(channel_mul=none, channel_add=none, relu=True)):
        assert F.linear(x, w, epilogue=F.Epilogue(**kw)).shape == (3, 0)
