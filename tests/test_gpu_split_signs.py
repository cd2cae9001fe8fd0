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
