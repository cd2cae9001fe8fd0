"""A run's batched sums and its unaries in the caller's buffer, against the
half-steps taken one by one (bit for bit)."""
import pytest
import torch

from cnn_crf_stereo_amd import ops
from cnn_crf_stereo_amd.capi import call, ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("iters", [0, 1, 31, 32, 33, 70])  # a batch holds 64 half-steps
def test_run_equals_half_steps(handle, iters):
    H, W, D = 7, 23, 16
    g = torch.Generator(device="cuda").manual_seed(iters)
    cost = -torch.softmax(3 * torch.randn((H, W, D), generator=g, device="cuda"), dim=2)
    wx, wy = torch.rand((2, H, W), generator=g, device="cuda")
    A = cost.clone()
    sums = torch.zeros(4 * iters + 1, dtype=torch.float64, device="cuda")
    for j in range(2 * iters):
        ops.slackprop_sweep(handle, cost, A, wx, wy, 0.5, 2.0, 2, 3 if j == 0 else j & 1, chain_sum=sums[j:],
                            kept_sum=sums[2 * iters + 1 + j:])
    labels = torch.empty((H, W), dtype=torch.int32, device="cuda")
    ops.slackprop_sweep(handle, cost, A, wx, wy, 0.5, 2.0, 2, 2, labels=labels, chain_sum=sums[2 * iters:])
    r = ops.slackprop(handle, cost, wx, wy, 0.5, 2.0, 2, iters, want_unaries=True)
    assert torch.equal(r["labels"], labels)
    assert torch.equal(r["unaries"], A)
    assert torch.equal(r["sums"], sums)
    lb = sums[2 * iters] + (sums[4 * iters] if iters else 0.0)
    assert r["lb"].item() == lb.item()
    # the unaries may replace the costs in place
    inplace = cost.clone()
    call("ccs_slackprop", handle.h, ptr(inplace), ptr(wx), ptr(wy), H, W, D, 0.5, 2.0, 2, iters, ptr(labels),
         ptr(inplace), None, None)
    assert torch.equal(inplace, A)
