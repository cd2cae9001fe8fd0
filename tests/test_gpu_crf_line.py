"""The three-wave sweep of few chains against the one-wave sweep of many, bit for
bit.

Chains are independent, so a row sweep of an image must leave what row sweeps of
its bands leave (and a column sweep what its vertical strips leave); the whole
image has more chains than the three-wave kernel takes, the bands have fewer.
"""
import pytest
import torch

from cnn_crf_stereo_amd import capi, ops

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 3, 8, 9, 10, 17, 24, 25, 26, 33, 34, 49, 57, 90]  # around the segments of 8 and blocks of 32 nodes


def bits(t):
    return t.contiguous().view(torch.int32)


@pytest.mark.parametrize("D", [2, 5, 32, 64, 66, 100, 128])
@pytest.mark.parametrize("n", LENGTHS)
def test_bands_equal_whole(handle, D, n):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    chains = 4 * cus + 3
    cuts = [0, 1, 40, 40 + cus + 1, chains - 2 * cus, chains]  # bands of 1 chain to 2 per CU
    for direction in (0, 1):
        H, W = (chains, n) if direction == 0 else (n, chains)
        g = torch.Generator(device="cuda").manual_seed(131 * D + n + direction)
        cost = -torch.softmax(3 * torch.randn((H, W, D), generator=g, device="cuda"), dim=2)
        cost[0, 0, D // 2 + 1:] = float("inf")
        A = cost + 0.1 * torch.randn((H, W, D), generator=g, device="cuda")
        wx, wy = torch.rand((2, H, W), generator=g, device="cuda")
        whole = A.clone()
        sums = torch.zeros(2, dtype=torch.float64, device="cuda")
        ops.slackprop_sweep(handle, cost, whole, wx, wy, 0.5, 2.0, 2, direction, chain_sum=sums[0:], kept_sum=sums[1:])
        got, total = [], torch.zeros_like(sums)
        for a, b in zip(cuts, cuts[1:]):
            cut = (lambda t: t[a:b].contiguous()) if direction == 0 else (lambda t: t[:, a:b].contiguous())
            band, s = cut(A), torch.zeros_like(sums)
            ops.slackprop_sweep(handle, cut(cost), band, cut(wx), cut(wy), 0.5, 2.0, 2, direction, chain_sum=s[0:],
                                kept_sum=s[1:])
            got.append(band)
            total += s
        got = torch.cat(got, dim=direction)
        assert torch.equal(torch.isnan(got), torch.isnan(whole))
        keep = ~torch.isnan(whole)
        assert torch.equal(bits(got[keep]), bits(whole[keep]))
        # the same per-chain values, summed in another order
        assert torch.allclose(total, sums, rtol=0, atol=chains * 2.0 ** -52 * float(chains * n))


@pytest.mark.parametrize("D", [2, 16, 17, 31, 32, 33])
@pytest.mark.parametrize("H,W", [(5, 1), (3, 2), (9, 40), (4, 77)])
def test_decode_ignores_infinite_labels(handle, D, H, W):
    """Labels and gaps of D labels, and of 64 of which all but D cost +inf."""
    g = torch.Generator(device="cuda").manual_seed(D + W)
    A = -torch.softmax(3 * torch.randn((H, W, D), generator=g, device="cuda"), dim=2)
    wx = torch.rand((H, W), generator=g, device="cuda")
    full = torch.full((H, W, 64), float("inf"), device="cuda")
    full[:, :, :D] = A
    got, want = (ops.slackprop_decode_gap(handle, x, wx, 0.5, 2.0, 2) for x in (A, full))
    assert torch.equal(got[0], want[0])
    assert torch.equal(bits(got[1]), bits(want[1]))


@pytest.mark.parametrize("D", [66, 128])
@pytest.mark.parametrize("H,W", [(7, 41), (300, 10), (1, 20), (20, 1)])
def test_per_edge_equals_element_path(handle, D, H, W):
    """Per-edge penalties; volumes off a lane's alignment take the element-wise kernel."""
    g = torch.Generator(device="cuda").manual_seed(D + W)
    base = -torch.softmax(3 * torch.randn((H, W, D), generator=g, device="cuda"), dim=2)
    pen = torch.rand((2, H, W, 2), generator=g, device="cuda")
    pen[0] += pen[1]  # P2 >= P1
    buf = torch.empty(base.numel() + 1, device="cuda")
    odd = buf[1:].view(base.shape).copy_(base)
    want = ops.slackprop_pw(handle, odd, pen, 2, 3)
    got = ops.slackprop_pw(handle, base, pen, 2, 3)
    assert torch.equal(got["labels"], want["labels"])
    assert torch.equal(got["sums"], want["sums"])


def test_streamed_costs_equal_kept_costs():
    """Volumes above the streaming size against bands below it."""
    H, W, D = 300, 1300, 100  # 156 MB; bands of 100 rows 52 MB
    g = torch.Generator(device="cuda").manual_seed(5)
    cost = -torch.softmax(3 * torch.randn((H, W, D), generator=g, device="cuda"), dim=2)
    wx, wy = torch.rand((2, H, W), generator=g, device="cuda")
    h = capi.Handle()
    whole = cost.clone()
    ops.slackprop_sweep(h, cost, whole, wx, wy, 0.5, 2.0, 2, 0)
    bands = cost.clone()
    for a in range(0, H, 100):
        s = slice(a, a + 100)
        ops.slackprop_sweep(h, cost[s], bands[s], wx[s], wy[s], 0.5, 2.0, 2, 0)
    assert torch.equal(bits(whole), bits(bands))
    ops.slackprop_sweep(h, cost, whole, wx, wy, 0.5, 2.0, 2, 1)
    for a in range(0, W, 260):
        s = slice(a, a + 260)
        c, b = cost[:, s].contiguous(), bands[:, s].contiguous()
        ops.slackprop_sweep(h, c, b, wx[:, s].contiguous(), wy[:, s].contiguous(), 0.5, 2.0, 2, 1)
        bands[:, s] = b
    assert torch.equal(bits(whole), bits(bands))
    h.close()
