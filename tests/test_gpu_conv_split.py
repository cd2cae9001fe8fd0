"""float32 layers on split 16-bit products: tile edges, value ranges, non-finite inputs.

A float16 pair holds a value to 2^-24 of itself and 2^-39 of its block's largest
value, and the products leave out 2^-24 |x w| more: 4 * 2^-24 |x w| in all; the
exact three-way split leaves out 2^-26 |x w|.  A 32-deep step has at most six
roundings at the size of its partial sums and the 30 steps one each, so |error|
<= 48 * 2^-24 * (sum |x w| + |b|).  The relative 2-norm is held to 3e-7: 30 random
roundings give about 1.5e-7, one missing partial product 1e-6 or more.
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from cnn_crf_stereo_amd import capi, ops

pytestmark = pytest.mark.gpu


def reference(x, w, b):
    """True convolution of planar float64 maps, and the sum of |x w| + |b|."""
    wf = torch.as_tensor(w).double().flip(2, 3)
    xd, bd = torch.as_tensor(x).double()[None], torch.as_tensor(b).double()
    return F.conv2d(xd, wf, bd)[0].numpy(), F.conv2d(xd.abs(), wf.abs(), bd.abs())[0].numpy()


def layer_out(handle, x, w, b):
    K, C = w.shape[:2]
    hwc = torch.zeros((*x.shape[1:], capi.feature_stride(C)), device="cuda")
    hwc[:, :, :C] = torch.as_tensor(x, device="cuda").permute(1, 2, 0)
    y = ops.ConvLayer(handle, w, b, "fp32", act=False)(handle, hwc)
    assert torch.count_nonzero(y[:, :, K:]).item() == 0, "padding channels must stay zero"
    return y[:, :, :K].permute(2, 0, 1).cpu().numpy()


@pytest.mark.parametrize("C,K,k,H,W,scale", [
    (100, 100, 3, 3, 3, 1.0),      # one output pixel
    (100, 100, 3, 18, 18, 1.0),    # exactly one tile
    (100, 100, 3, 19, 35, 1.0),    # one row and one column over
    (100, 100, 2, 17, 16, 1.0),    # a full-height tile, one column short
    (100, 100, 2, 40, 150, 1e15),  # several tiles, large values
    (97, 104, 3, 21, 40, 1e-20),   # the fewest inputs and most outputs of the stride, small values
    (64, 64, 3, 19, 35, 1.0),
    (57, 64, 3, 18, 20, 1.0),
])
def test_split_layer(handle, C, K, k, H, W, scale):
    rng = np.random.default_rng(C + K + k + H)
    x = (scale * rng.uniform(-1, 1, (C, H, W))).astype(np.float32)
    a = np.sqrt(6.0 / (2 * C * k * k))
    w = rng.uniform(-a, a, (K, C, k, k)).astype(np.float32)
    b = (scale * rng.uniform(-0.1, 0.1, K)).astype(np.float32)
    ref, size = reference(x, w, b)
    got = layer_out(handle, x, w, b).astype(np.float64)
    assert np.all(np.abs(got - ref) <= 48 * 2.0**-24 * size)
    assert np.linalg.norm(got - ref) <= 3e-7 * np.linalg.norm(ref)


@pytest.mark.parametrize("C,k", [(100, 3), (100, 2), (64, 3)])
def test_split_layer_of_uneven_pixels(handle, C, k):
    """Pixels and output channels of sizes 1e-12 to 1e12 side by side: every
    output keeps the precision of its own terms."""
    rng = np.random.default_rng(C + 7 * k)
    x = (rng.uniform(-1, 1, (C, 20, 37)) * 10.0 ** rng.uniform(-12, 12, (1, 20, 37))).astype(np.float32)
    w = (rng.uniform(-0.1, 0.1, (C, C, k, k)) * 10.0 ** rng.uniform(-12, 12, (C, 1, 1, 1))).astype(np.float32)
    b = np.zeros(C, np.float32)
    ref, size = reference(x, w, b)
    got = layer_out(handle, x, w, b).astype(np.float64)
    assert np.all(np.abs(got - ref) <= 48 * 2.0**-24 * size)


@pytest.mark.parametrize("C,k", [(100, 3), (100, 2), (64, 3)])
def test_split_layer_keeps_infinities_and_nan(handle, C, k):
    """An infinity keeps its sign through every weight (0.5 and 300 split with
    zero and opposite-sign residuals), a NaN stays NaN, and the largest finite
    values, which round to infinity in bf16, stay finite."""
    rng = np.random.default_rng(C + k)
    x = rng.uniform(-1, 1, (C, 20, 37)).astype(np.float32)
    w = rng.uniform(-0.1, 0.1, (C, C, k, k)).astype(np.float32)
    w[0], w[1], w[2] = 0.5, 300.7, -0.25
    w[:, 7] = 0.001
    b = np.zeros(C, np.float32)
    x[3, 4, 5], x[5, 12, 20], x[6, 2, 30] = np.inf, -np.inf, np.nan
    x[7, 15, 8] = np.finfo(np.float32).max
    ref, size = reference(x, w, b)
    got = layer_out(handle, x, w, b).astype(np.float64)
    fin = np.isfinite(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[~fin & ~np.isnan(ref)], ref[~fin & ~np.isnan(ref)])
    assert np.all(np.abs(got[fin] - ref[fin]) <= 48 * 2.0**-24 * size[fin])
