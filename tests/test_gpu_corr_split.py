"""float32 correlation on split float16 products: pixel tiles, windows, channel
remainders, non-finite features.

A float16 pair holds a value to 2^-24 of itself and 2^-39 of the largest of its
pixel's 32 channels, and the products leave out 2^-24 |ab|: 4 * 2^-24 |ab| in all.
A stage takes at most 4 roundings and at most 8 stages follow, so |error| <=
16 * 2^-24 * sum |a b|.
"""
import numpy as np
import pytest
import torch

from cnn_crf_stereo_amd import capi, ops

pytestmark = pytest.mark.gpu


def volumes(handle, f0, f1, dmin, step, D):
    H, W, C = f0.shape
    Cs = capi.feature_stride(C)
    dev = []
    for f in (f0, f1):
        t = torch.zeros((H, W, Cs), device="cuda")
        t[:, :, :C] = torch.as_tensor(f)
        dev.append(t)
    got = ops.correlation_volume(handle, dev[0], dev[1], C, dmin, step, D, epilogue="raw").double().cpu().numpy()
    # (a column outside the image counts as a pixel of zeros)
    a, far = f0.astype(np.float64), W + abs(dmin) + D * abs(step)
    b = np.pad(f1.astype(np.float64), ((0, 0), (far, far), (0, 0)))
    ref, size = np.zeros((H, W, D)), np.zeros((H, W, D))
    for k in range(D):
        q = b[:, far - (dmin + k * step):][:, :W]
        with np.errstate(invalid="ignore"):
            ref[:, :, k], size[:, :, k] = (a * q).sum(-1), np.abs(a * q).sum(-1)
    return got, ref, size


@pytest.mark.parametrize("H,W,C,dmin,step,D", [
    (1, 1, 8, 0, 1, 1),
    (2, 17, 100, 0, 1, 16),      # one pixel over a wave
    (2, 129, 100, 3, 1, 32),     # one over a tile, window of 3 blocks
    (1, 150, 64, 0, 2, 30),      # every other column
    (1, 300, 100, 0, 1, 64),     # 5 blocks
    (1, 140, 36, 0, -1, 70),     # the other way, channels past the last 32
    (1, 260, 100, 0, 1, 128),    # 9 blocks
    (2, 300, 100, 0, 1, 256),    # 17 blocks, the tile of 64 pixels
    (1, 65, 256, 0, 1, 40),      # 8 stages
])
def test_correlation(handle, H, W, C, dmin, step, D):
    rng = np.random.default_rng(H + W + C + D)
    f0, f1 = (rng.normal(size=(H, W, C)).astype(np.float32) for _ in range(2))
    f0 *= (10.0 ** rng.uniform(-12, 12, (H, W, 1))).astype(np.float32)  # pixels of any size side by side
    got, ref, size = volumes(handle, f0, f1, dmin, step, D)
    assert np.all(np.abs(got - ref) <= 16 * 2.0**-24 * size)


def test_non_finite_features(handle):
    rng = np.random.default_rng(4)
    f0, f1 = (rng.uniform(0.1, 1, (2, 150, 100)).astype(np.float32) for _ in range(2))
    f0[0, 20, 3], f0[1, 70, 99], f1[0, 100, 40] = np.inf, np.nan, -np.inf
    got, ref, size = volumes(handle, f0, f1, 0, 1, 48)
    fin = np.isfinite(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = ~fin & ~np.isnan(ref)
    assert np.array_equal(got[inf], ref[inf])
    assert np.all(np.abs(got[fin] - ref[fin]) <= 16 * 2.0**-24 * size[fin])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("W,dmin,step,D", [
    (150, 0, 1, 128), (70, 3, 1, 112), (150, 0, -1, 127),  # in the accumulators, 9 column tiles
    (150, 0, 1, 111),                                      # the widest band that goes through LDS
    (300, 0, 1, 256), (66, 0, 1, 240),                     # 17 column tiles
])
def test_softmax_epilogue(handle, dtype, W, dmin, step, D):
    """-softmax of the raw volume, which the raw epilogue gives: exp(s - max) has
    2^-21 (the hardware's exp2 and the rounding of its argument, |s - max| < 16), the
    sum D more roundings at most, the quotient three."""
    g = torch.Generator(device="cuda").manual_seed(W + D)
    f0, f1 = (torch.randn((3, W, 104), generator=g, device="cuda").mul(0.3).to(dtype) for _ in range(2))
    raw = ops.correlation_volume(handle, f0, f1, 104, dmin, step, D, epilogue="raw").double()
    got = ops.correlation_volume(handle, f0, f1, 104, dmin, step, D).double()
    want = -torch.softmax(raw, dim=-1)
    tol = (2.0**-20 + (D + 3) * 2.0**-24) * want.abs() + 1e-30
    assert ((got - want).abs() <= tol).all()
