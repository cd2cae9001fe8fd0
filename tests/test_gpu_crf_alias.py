"""unaries_out may lie over an input of a CRF run: the run reads its inputs as they were."""
import pytest
import torch

from cnn_crf_stereo_amd import capi, ops
from cnn_crf_stereo_amd.capi import call, ptr

pytestmark = pytest.mark.gpu

H, W, D, ITERS = 30, 44, 24, 3


def tensors(n_weights):
    g = torch.Generator(device="cuda").manual_seed(1)
    cost = -torch.softmax(3 * torch.randn((H, W, D), generator=g, device="cuda"), dim=2)
    return cost, [torch.rand((H, W), generator=g, device="cuda") + 0.1 for _ in range(n_weights)]


def outputs():
    return (torch.empty((H, W), dtype=torch.int32, device="cuda"),
            torch.zeros(4 * ITERS + 1, dtype=torch.float64, device="cuda"),
            torch.zeros(1, dtype=torch.float64, device="cuda"))


@pytest.mark.parametrize("over", ["cost", "wx", "wy"])
def test_weights(handle, over):
    cost, (wx, wy) = tensors(2)
    want = ops.slackprop(handle, cost, wx, wy, 0.5, 2.0, 2, ITERS, want_unaries=True)
    out = torch.zeros((H, W, D), device="cuda")
    inside = out if over == "cost" else out.flatten()[100:100 + H * W].view(H, W)
    inside.copy_(dict(cost=cost, wx=wx, wy=wy)[over])
    use = dict(dict(cost=cost, wx=wx, wy=wy), **{over: inside})
    labels, sums, lb = outputs()
    call("ccs_slackprop", handle.h, ptr(use["cost"]), ptr(use["wx"]), ptr(use["wy"]), H, W, D, 0.5, 2.0, 2, ITERS,
         ptr(labels), ptr(out), ptr(sums), ptr(lb))
    for got, key in ((labels, "labels"), (sums, "sums"), (lb, "lb"), (out, "unaries")):
        assert torch.equal(got, want[key]), key


def test_penalties(handle):
    cost, (a, b, c, d) = tensors(4)
    pen, _ = ops.pairwise_penalties(handle, torch.stack([a, b, a + c, b + d]))
    want = ops.slackprop_pw(handle, cost, pen, 2, ITERS, want_unaries=True)
    out = torch.zeros((H, W, D), device="cuda")
    inside = out.flatten()[64:64 + pen.numel()].view(pen.shape)
    inside.copy_(pen)
    labels, sums, lb = outputs()
    call("ccs_slackprop_pw", handle.h, ptr(cost), ptr(inside), pen.shape[0], H, W, D, 2, ITERS, ptr(labels), ptr(out),
         ptr(sums), ptr(lb))
    for got, key in ((labels, "labels"), (sums, "sums"), (lb, "lb"), (out, "unaries")):
        assert torch.equal(got, want[key]), key
