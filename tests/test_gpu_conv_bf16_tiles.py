"""The bf16 100-channel layers on 32- and 64-pixel tiles: the widths and heights
at which a tile is full, over or short, and both sides of the rule between them.

Products of bfloat16 values are exact in the matrix core and 900 of them are
summed in float32 (2^-24 each at the size of the whole), then rounded to
bfloat16 (8 significant bits): |error| <= 2^-24 * 900 * sum |x w| + 2^-8 |y|.
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from cnn_crf_stereo_amd import capi, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [3, 2])
@pytest.mark.parametrize("Ho,Wo", [
    (1, 1), (4, 32), (5, 33), (3, 31), (9, 65),  # edges of the narrow tile
    (190, 626),  # one round of 48 x 10 wide tiles, two of 48 x 20 narrow ones (256 CUs)
    (190, 200),  # one round of either: narrow
])
def test_tiles(handle, k, Ho, Wo):
    C = 100
    g = torch.Generator(device="cuda").manual_seed(Ho + Wo + k)
    x = torch.randn((C, Ho + k - 1, Wo + k - 1), generator=g, device="cuda").bfloat16()
    w = (torch.rand((C, C, k, k), generator=g, device="cuda") - 0.5).mul(0.1).bfloat16().float()
    b = torch.rand(C, generator=g, device="cuda") - 0.5
    hwc = torch.zeros((Ho + k - 1, Wo + k - 1, capi.feature_stride(C)), device="cuda", dtype=torch.bfloat16)
    hwc[:, :, :C] = x.permute(1, 2, 0)
    y = ops.ConvLayer(handle, w.cpu().numpy(), b.cpu().numpy(), "bf16", act=False)(handle, hwc)
    assert y.shape[:2] == (Ho, Wo)
    assert torch.count_nonzero(y[:, :, C:]).item() == 0
    got = y[:, :, :C].permute(2, 0, 1).double().cpu().numpy()
    xd, wd, bd = x.double().cpu()[None], w.double().cpu().flip(2, 3), b.double().cpu()
    ref, size = F.conv2d(xd, wd, bd)[0].numpy(), F.conv2d(xd.abs(), wd.abs(), bd.abs())[0].numpy()
    assert np.all(np.abs(got - ref) <= 2.0**-24 * 900 * size + 2.0**-8 * np.abs(ref) * (1 + 2.0**-8))
