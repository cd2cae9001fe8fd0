"""Label counts that fill whole lanes but not the wave: the vector path against
the element-wise one, bit for bit.

Volumes whose base is not aligned to a lane's labels take the element-wise
path, so the same run on a view shifted by one float must give the same bits.
"""
import pytest
import torch

from cnn_crf_stereo_amd import ops

pytestmark = pytest.mark.gpu


def shifted(t):
    """A contiguous copy of t that starts one float after an aligned address."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    view = buf[1:].view(t.shape)
    return view.copy_(t)


def run(h, cost, wx, wy, A, iters):
    H, W, D = cost.shape
    sums = torch.zeros((2, 2 * iters + 1), dtype=torch.float64, device="cuda")
    for j in range(2 * iters):
        ops.slackprop_sweep(h, cost, A, wx, wy, 0.5, 2.0, 2, 3 if j == 0 else j & 1, chain_sum=sums[0, j:],
                            kept_sum=sums[1, j:])
    unaries = A.clone()
    labels = torch.empty((H, W), dtype=torch.int32, device="cuda")
    ops.slackprop_sweep(h, cost, A, wx, wy, 0.5, 2.0, 2, 2, labels=labels, chain_sum=sums[0, 2 * iters:])
    return unaries, labels, sums


@pytest.mark.parametrize("D", [66, 70, 100, 126, 132, 200, 252])  # 2 and 4 labels per lane
@pytest.mark.parametrize("H,W", [(5, 40), (37, 3), (1, 30), (30, 1)])
def test_lane_path_equals_element_path(handle, D, H, W):
    g = torch.Generator(device="cuda").manual_seed(D + W)
    cost = -torch.softmax(3 * torch.randn((H, W, D), generator=g, device="cuda"), dim=2)
    cost[0, 0, :3] = float("inf")
    wx, wy = torch.rand((2, H, W), generator=g, device="cuda")
    want = run(handle, shifted(cost), wx, wy, shifted(cost), 3)
    got = run(handle, cost, wx, wy, torch.empty_like(cost), 3)
    for a, b in zip(got, want):  # (an infinite cost leaves NaN unaries: inf - inf)
        assert torch.allclose(a, b, rtol=0, atol=0, equal_nan=True)
