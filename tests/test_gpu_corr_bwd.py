"""The correlation adjoint on split products, at the edges of its tiles and
chunks, against float64.

Products are exact (float32 maps: but for 2^-26 of each); a 32-deep step rounds
at most six times at the size of its partial sums, the at most
3 ceil(D / 64) + 2 steps once each more, so
|error| <= (14 + 9 ceil(D / 64)) 2^-24 sum |G F|, and bfloat16 maps round the
result to 2^-8 (half a unit of its eighth significant bit).
"""
import pytest
import torch

from cnn_crf_stereo_amd import capi, ops

pytestmark = pytest.mark.gpu


def reference(f0, f1, G, dmin, step):
    """df0, df1 and the sums of |G F| in float64 (H x W x C maps)."""
    f0, f1, G = f0.double(), f1.double(), G.double()
    W = f0.shape[1]
    out = [torch.zeros_like(f0) for _ in range(4)]
    for k in range(G.shape[2]):
        d = dmin + k * step  # column w of f0 meets column w - d of f1
        lo, hi = max(d, 0), min(W, W + d)
        if lo >= hi:
            continue
        g, a, b = G[:, lo:hi, k, None], f0[:, lo:hi], f1[:, lo - d:hi - d]
        out[0][:, lo:hi] += g * b
        out[1][:, lo - d:hi - d] += g * a
        out[2][:, lo:hi] += (g * b).abs()
        out[3][:, lo - d:hi - d] += (g * a).abs()
    return out


def maps(g, H, W, C, dtype):
    f = torch.zeros((H, W, capi.feature_stride(C)), device="cuda")
    f[:, :, :C] = torch.tanh(torch.randn((H, W, C), generator=g, device="cuda"))
    return f.to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,W,D,dmin,step,C", [
    (1, 1, 1, 0, 1, 100),
    (2, 127, 64, 0, 1, 100),     # one tile, a pixel short
    (9, 128, 65, 0, 1, 100),     # one tile, a disparity over (float32) chunk
    (3, 129, 128, 3, 1, 100),    # a pixel over
    (2, 300, 129, 0, 1, 100),    # a disparity over the bfloat16 chunk
    (1, 400, 256, 0, 1, 100),
    (2, 40, 100, 0, 1, 100),     # the band is wider than the image
    (2, 150, 33, -20, 1, 65),    # both signs of the offset, fewest channels
    (2, 150, 40, 5, -1, 112),    # decreasing disparities, most channels
])
def test_corr_adjoint(handle, H, W, D, dmin, step, C, dtype):
    g = torch.Generator(device="cuda").manual_seed(W + D)
    f0, f1 = maps(g, H, W, C, dtype), maps(g, H, W, C, dtype)
    G = torch.randn((H, W, D), generator=g, device="cuda") * torch.rand((H, W, 1), generator=g, device="cuda") ** 8
    r0, r1, s0, s1 = reference(f0, f1, G, dmin, step)
    d0, d1 = ops.correlation_volume_backward(handle, f0, f1, C, dmin, step, D, G)
    for d, r, s in ((d0, r0, s0), (d1, r1, s1)):
        tol = (14 + 9 * ((D + 63) // 64)) * 2.0**-24 * s
        if dtype == torch.bfloat16:
            tol = tol + 2.0**-8 * (r.abs() + tol)
        assert ((d.double() - r).abs() <= tol).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_corr_adjoint_non_finite_gradient(handle, dtype):
    """An infinite or NaN gradient reaches the pixels it belongs to and no other."""
    H, W, D, C = 2, 200, 70, 100
    g = torch.Generator(device="cuda").manual_seed(3)
    f0, f1 = maps(g, H, W, C, dtype), maps(g, H, W, C, dtype)
    G = torch.randn((H, W, D), generator=g, device="cuda")
    G[0, 100, 3], G[0, 150, 69], G[1, 130, 40] = float("inf"), float("-inf"), float("nan")
    G[1, 90, 10] = 3.4e38
    r0, r1, _, _ = reference(f0, f1, G, 0, 1)
    d0, d1 = ops.correlation_volume_backward(handle, f0, f1, C, 0, 1, D, G)
    for d, r in ((d0, r0), (d1, r1)):
        d = d.double()
        assert torch.equal(d.isnan(), r.isnan())
        assert torch.equal(d.isposinf(), r.isposinf()) and torch.equal(d.isneginf(), r.isneginf())
