"""Chains too long for the three-wave kernel to hold as many as the one-wave kernel: an
image of more chains than that against bands of few, bit for bit."""
import pytest
import torch

from cnn_crf_stereo_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("direction,chains,n,D", [
    (0, 300, 4200, 8), (0, 300, 3000, 66), (1, 300, 3400, 16), (1, 1000, 1300, 16), (1, 300, 2600, 66),
])
def test_bands_equal_whole(handle, direction, chains, n, D):
    H, W = (chains, n) if direction == 0 else (n, chains)
    g = torch.Generator(device="cuda").manual_seed(n + D)
    cost = torch.randn((H, W, D), generator=g, device="cuda")
    A = cost + 0.1 * torch.randn((H, W, D), generator=g, device="cuda")
    wx, wy = torch.rand((2, H, W), generator=g, device="cuda")
    whole, parts = A.clone(), []
    ops.slackprop_sweep(handle, cost, whole, wx, wy, 0.5, 2.0, 2, direction)
    for a in range(0, chains, 200):
        cut = (lambda t: t[a:a + 200].contiguous()) if direction == 0 else (lambda t: t[:, a:a + 200].contiguous())
        band = cut(A)
        ops.slackprop_sweep(handle, cut(cost), band, cut(wx), cut(wy), 0.5, 2.0, 2, direction)
        parts.append(band)
    assert torch.equal(torch.cat(parts, dim=direction).view(torch.int32), whole.view(torch.int32))
