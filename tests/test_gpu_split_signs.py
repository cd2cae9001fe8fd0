"""The split products' errors have no common sign, also in the correlation's scores and
in weight gradients of one segment per workgroup.

The matrix unit rounds its 16-bit products' sums down.  For N outputs with independent
errors of zero mean and root mean square r, the mean error stays within 5 r / sqrt(N)
for each of some hundred groups; weight gradients share the rounded inputs of 9 taps,
which widens that by at most sqrt(9).
"""
import numpy as np
import pytest
import torch

from cnn_crf_stereo_amd import capi, ops

pytestmark = pytest.mark.gpu


def bias(got, ref):
    """The largest mean error of a group (groups x outputs), in units of r / sqrt(N)."""
    err = got.double().cpu().reshape(ref.shape) - ref
    rms = err.square().mean(dim=1).sqrt()
    return (err.mean(dim=1).abs() / (rms + 1e-300) * np.sqrt(err.shape[1])).max().item()


def maps(g, H, W, C=100):
    x = torch.zeros((H, W, capi.feature_stride(C)))
    x[:, :, :C] = torch.rand((H, W, C), generator=g) * 2 - 1
    return x


@pytest.mark.parametrize("W,D,step", [(300, 32, 1), (260, 100, 1), (200, 64, -1), (280, 200, 1)])
def test_correlation(handle, W, D, step):
    g = torch.Generator().manual_seed(W)
    H, C = 90, 100
    f0, f1 = maps(g, H, W), maps(g, H, W)
    got = ops.correlation_volume(handle, f0.cuda(), f1.cuda(), C, 0, step, D, epilogue="raw").cpu()
    a, b = f0[:, :, :C].double(), f1[:, :, :C].double()
    lo, hi = (D - 1, W) if step > 0 else (0, W - D + 1)  # pixels whose whole band is inside the image
    ref = torch.stack([(a[:, lo:hi] * b[:, lo - step * d:hi - step * d]).sum(-1).flatten() for d in range(D)])
    assert bias(got[:, lo:hi].permute(2, 0, 1), ref) <= 5


@pytest.mark.parametrize("k,H", [(3, 74), (3, 40), (2, 110)])
def test_weight_gradient_of_one_segment_per_workgroup(handle, k, H):
    """A map of 32 output pixels per row and no more rows than workgroups: the signs
    alternate over the map's segments, not over a workgroup's."""
    g = torch.Generator().manual_seed(k)
    C, W = 100, 31 + k
    Ho, Wo = H - k + 1, W - k + 1
    x, dz = maps(g, H, W), maps(g, Ho, Wo)
    w = torch.zeros((C, C, k, k), device="cuda")
    _, dw, _ = ops.conv2d_backward_stored(handle, x.cuda(), torch.zeros((Ho, Wo, 104), device="cuda"), w, dz.cuda(),
                                          act=False)
    z = dz[:, :, :C].double().reshape(-1, C)
    ref = torch.stack([z.t() @ x[k - 1 - a:k - 1 - a + Ho, k - 1 - b:k - 1 - b + Wo, :C].double().reshape(-1, C)
                       for a in range(k) for b in range(k)], dim=2)
    assert bias(dw.reshape(1, -1), ref.reshape(1, -1)) <= 15


def offset(got, ref):
    """The largest mean error of a group (groups x outputs), in units of its root mean square."""
    err = got.double().cpu().reshape(ref.shape) - ref
    return (err.mean(dim=1).abs() / ref.square().mean(dim=1).sqrt()).max().item()


@pytest.mark.parametrize("C,k", [(100, 3), (100, 2), (64, 3)])
@pytest.mark.parametrize("H,W", [(131, 166), (250, 203)])
def test_layer_of_positive_maps(handle, C, k, H, W):
    """Inputs with a mean: what rounding leaves out of a weight is the same for every
    pixel, but the weights of a row together leave out nothing.  A float32 output is
    itself off by up to 2^-24; the mean over a map stays within half of that."""
    g = torch.Generator().manual_seed(C + k + H)
    x = maps(g, H, W, C).abs()
    w = (torch.rand((C, C, k, k), generator=g) * 2 - 1) * 0.1
    got = ops.ConvLayer(handle, w.numpy(), np.zeros(C, np.float32), "fp32", act=False)(handle, x.cuda())[:, :, :C]
    ref = torch.nn.functional.conv2d(x[:, :, :C].double().permute(2, 0, 1)[None], w.double().flip(2, 3))[0].reshape(C, -1)
    assert offset(got.permute(2, 0, 1), ref) <= 2.0**-25
    # the input gradient, whose filters are the adjoint ones
    dy = maps(g, H - k + 1, W - k + 1, C).abs()
    dx, _, _ = ops.conv2d_backward_stored(handle, x.cuda(), torch.zeros_like(dy).cuda(), w.cuda(), dy.cuda(), act=False)
    ref = torch.nn.functional.conv_transpose2d(dy[:, :, :C].double().permute(2, 0, 1)[None], w.double().flip(2, 3))
    assert offset(dx[:, :, :C].permute(2, 0, 1), ref[0].reshape(C, -1)) <= 2.0**-25
