"""The image layer on split bf16 products: shares of pixels, channel remainders,
planes, non-finite inputs.

Six products of exactly split terms leave out less than 2^-26 |x w|; the matrix
core rounds at most once per product set and the bias once more, so |error| <=
8 * 2^-24 * (sum |x w| + |b|), plus half a bfloat16 unit (8 significant bits: 2^-8) for bf16 maps; a
wrong tap or a missing product is 2^-17 of a term or more.
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from cnn_crf_stereo_amd import ops

pytestmark = pytest.mark.gpu


def check(handle, x, w, b, precision):
    K = w.shape[0]
    xd, wd, bd = (torch.as_tensor(v).double() for v in (x, w, b))
    ref = F.conv2d(xd[None], wd.flip(2, 3), bd)[0].numpy()
    size = F.conv2d(xd.abs()[None], wd.abs().flip(2, 3), bd.abs())[0].numpy()
    y = ops.ConvLayer(handle, w, b, precision, act=False)(handle, torch.as_tensor(x, device="cuda"), layout="nchw")
    assert torch.count_nonzero(y[:, :, K:]).item() == 0, "padding channels must stay zero"
    got = y[:, :, :K].permute(2, 0, 1).double().cpu().numpy()
    fin = np.isfinite(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = ~fin & ~np.isnan(ref)
    assert np.array_equal(got[inf], ref[inf])
    bound = 8 * 2.0**-24 * size + (2.0**-8 * np.abs(ref) * (1 + 2.0**-8) if precision == "bf16" else 0)
    assert np.all(np.abs(got[fin] - ref[fin]) <= bound[fin])


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("C,K,H,W", [
    (3, 100, 3, 3),      # one output pixel
    (3, 97, 3, 18),      # exactly one share of 16 pixels
    (2, 112, 4, 19),     # pixels over two rows of one share
    (3, 64, 5, 40),
    (2, 49, 37, 61),
    (3, 104, 190, 203),  # two shares and more per wave
])
def test_image_layer(handle, precision, C, K, H, W):
    rng = np.random.default_rng(C + K + H)
    x = rng.normal(size=(C, H, W)).astype(np.float32)
    w = rng.uniform(-0.3, 0.3, (K, C, 3, 3)).astype(np.float32)
    b = rng.uniform(-0.1, 0.1, K).astype(np.float32)
    check(handle, x, w, b, precision)


def test_large_gray_image(handle):
    rng = np.random.default_rng(1)
    x = rng.normal(size=(1, 513, 511)).astype(np.float32)
    check(handle, x, rng.uniform(-0.3, 0.3, (100, 1, 3, 3)).astype(np.float32), np.zeros(100, np.float32), "fp32")


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_non_finite_pixels(handle, precision):
    rng = np.random.default_rng(2)
    x = rng.normal(size=(3, 20, 37)).astype(np.float32)
    w = rng.uniform(0.1, 0.3, (100, 3, 3, 3)).astype(np.float32) * np.where(np.arange(100) % 2, 1, -1)[:, None, None, None]
    x[0, 4, 5], x[1, 12, 20], x[2, 2, 30] = np.inf, -np.inf, np.nan
    check(handle, x, w.astype(np.float32), np.zeros(100, np.float32), precision)
