"""The split products' errors have no common sign: sums over a map gather none.

The matrix unit rounds its 16-bit products' sums down; uncorrected, every output
is off by a share of its rounding error in the same direction.  For N outputs
with independent errors of zero mean and root mean square r, the mean error
stays within 4 r / sqrt(N) for each of some hundred channels; neighbouring outputs
share the rounded inputs of up to KH * KW = 9 taps, which widens that by at most
sqrt(9): |mean| <= 12 r / sqrt(N).
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from cnn_crf_stereo_amd import capi, ops

pytestmark = pytest.mark.gpu


def check(got, ref):
    """got, ref: channels x outputs."""
    err = got.double().cpu().reshape(ref.shape) - ref
    rms = err.square().mean(dim=1).sqrt()
    t = err.mean(dim=1).abs() / (rms + 1e-300) * np.sqrt(err.shape[1])
    assert t.max().item() <= 12, t.max().item()


def planar(t, C):
    return t[:, :, :C].permute(2, 0, 1).reshape(C, -1)


def maps(g, C, H, W):
    x = torch.zeros((H, W, capi.feature_stride(C)))
    x[:, :, :C] = torch.rand((H, W, C), generator=g) * 2 - 1
    return x


@pytest.mark.parametrize("C,k", [(100, 3), (100, 2), (64, 3)])
@pytest.mark.parametrize("H,W", [(74, 97), (131, 166)])
def test_layer_and_adjoint(handle, C, k, H, W):
    g = torch.Generator().manual_seed(C + k + H)
    x, y, dy = maps(g, C, H, W), maps(g, C, H - k + 1, W - k + 1), maps(g, C, H - k + 1, W - k + 1)
    w = (torch.rand((C, C, k, k), generator=g) * 2 - 1) * 0.1
    got = ops.ConvLayer(handle, w.numpy(), np.zeros(C, np.float32), "fp32", act=False)(handle, x.cuda())
    xd, wf = x[:, :, :C].double().permute(2, 0, 1), w.double().flip(2, 3)
    check(planar(got, C), F.conv2d(xd[None], wf)[0].reshape(C, -1))
    dx, dw, _ = ops.conv2d_backward_stored(handle, x.cuda(), y.cuda(), w.cuda(), dy.cuda(), act=False)
    dz = dy[:, :, :C].double().permute(2, 0, 1)
    check(planar(dx, C), F.conv_transpose2d(dz[None], wf)[0].reshape(C, -1))
    if C == 100:
        ref = F.conv2d(xd[:, None], dz[:, None]).flip(2, 3).transpose(0, 1)
        check(dw.reshape(C, -1), ref.reshape(C, -1))


@pytest.mark.parametrize("C,K", [(3, 100), (2, 64)])
def test_image_layer(handle, C, K):
    g = torch.Generator().manual_seed(C)
    x = torch.rand((C, 94, 203), generator=g) * 2 - 1
    w = torch.rand((K, C, 3, 3), generator=g) - 0.5
    got = ops.ConvLayer(handle, w.numpy(), np.zeros(K, np.float32), "fp32", act=False)(handle, x.cuda(), layout="nchw")
    check(planar(got, K), F.conv2d(x.double()[None], w.double().flip(2, 3))[0].reshape(K, -1))


@pytest.mark.parametrize("W,D", [(150, 32), (203, 100)])
def test_correlation_adjoint(handle, W, D):
    g = torch.Generator().manual_seed(W)
    H, C = 40, 100
    f0, f1, G = maps(g, C, H, W), maps(g, C, H, W), torch.rand((H, W, D), generator=g) - 0.5
    d0, d1 = ops.correlation_volume_backward(handle, f0.cuda(), f1.cuda(), C, 0, 1, D, G.cuda())
    r0, r1 = torch.zeros((H, W, C), dtype=torch.float64), torch.zeros((H, W, C), dtype=torch.float64)
    for d in range(D):
        Gd = G[:, d:, d, None].double()
        r0[:, d:] += Gd * f1[:, : W - d, :C].double()
        r1[:, : W - d] += Gd * f0[:, d:, :C].double()
    check(planar(d0, C), planar(r0, C))
    check(planar(d1, C), planar(r1, C))
