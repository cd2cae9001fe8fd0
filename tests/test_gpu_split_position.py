"""float32 kernels give equal inputs equal outputs, to the bit, wherever they lie in a
map: a layer of a crop is the crop of the layer, whatever the parity of its corner."""
import numpy as np
import pytest
import torch

from cnn_crf_stereo_amd import capi, ops

pytestmark = pytest.mark.gpu

CORNERS = [(0, 1), (1, 0), (3, 2), (8, 17)]


def maps(g, H, W, C=100):
    x = torch.zeros((H, W, capi.feature_stride(C)))
    x[:, :, :C] = torch.rand((H, W, C), generator=g) * 2 - 1
    return x.cuda()


@pytest.mark.parametrize("C,k", [(100, 3), (100, 2), (64, 3)])
@pytest.mark.parametrize("H,W", [(30, 45), (131, 166)])  # tiles of four rows and of eight
def test_layer(handle, C, k, H, W):
    g = torch.Generator().manual_seed(C + k)
    x = maps(g, H, W, C)
    w = (torch.rand((C, C, k, k), generator=g) - 0.5).numpy() * 0.2
    layer = ops.ConvLayer(handle, w, np.zeros(C, np.float32), "fp32", act=False)
    whole = layer(handle, x)
    for i, j in CORNERS:
        assert torch.equal(layer(handle, x[i:, j:].contiguous()), whole[i:, j:]), (i, j)


@pytest.mark.parametrize("C,K,H,W", [(3, 100, 40, 61), (2, 64, 40, 61), (1, 100, 560, 530)])
def test_image_layer(handle, C, K, H, W):
    g = torch.Generator().manual_seed(C)
    x = (torch.rand((C, H, W), generator=g) * 2 - 1).cuda()
    layer = ops.ConvLayer(handle, (torch.rand((K, C, 3, 3), generator=g) - 0.5).numpy(), np.zeros(K, np.float32), "fp32")
    whole = layer(handle, x, layout="nchw")
    for i, j in CORNERS:
        assert torch.equal(layer(handle, x[:, i:, j:].contiguous(), layout="nchw"), whole[i:, j:]), (i, j)


@pytest.mark.parametrize("D", [32, 128])
def test_correlation(handle, D):
    g = torch.Generator().manual_seed(D)
    f0, f1 = maps(g, 12, 260), maps(g, 12, 260)
    whole = ops.correlation_volume(handle, f0, f1, 100, 0, 1, D, epilogue="raw")
    for i, j in CORNERS:
        a, b = f0[i:, j:].contiguous(), f1[i:, j:].contiguous()
        part = ops.correlation_volume(handle, a, b, 100, 0, 1, D, epilogue="raw")
        assert torch.equal(part[:, D:], whole[i:, j + D:]), (i, j)


def test_correlation_adjoint_rows(handle):
    """(Along a row the terms are summed in an order that depends on the place.)"""
    g = torch.Generator().manual_seed(1)
    f0, f1, G = maps(g, 12, 150), maps(g, 12, 150), (torch.rand((12, 150, 40), generator=g) - 0.5).cuda()
    whole = ops.correlation_volume_backward(handle, f0, f1, 100, 0, 1, 40, G)
    for i in (1, 2, 5):
        part = ops.correlation_volume_backward(handle, f0[i:].contiguous(), f1[i:].contiguous(), 100, 0, 1, 40,
                                               G[i:].contiguous())
        assert all(torch.equal(p, w[i:]) for p, w in zip(part, whole)), i
