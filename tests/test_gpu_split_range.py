"""float32 kernels on split products keep float32's precision for every input: values
of any sizes inside one block of a common scale, and sums near the largest float.

Every case has outputs whose terms are small beside other values of their block,
which meet a zero.  A pair must hold each value to 2^-22 of itself or leave the block
to float32 products, whose chain of N additions is off by 2^-24 sqrt(N / 6) of the
sum's 2-norm (partial sums grow with sqrt(i / N), roundings are uniform): 3.7e-7 for
the 234 steps of a 3x3 layer, 4.5e-7 with 2^-22 / sqrt(12) per factor beside it.  The
2-norm of each output channel's error is held to 8e-7 of the channel's.
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from cnn_crf_stereo_amd import capi, ops

pytestmark = pytest.mark.gpu


def uniform(rng, *shape):
    """Magnitudes of one size: in (-1, 1) without what lies near zero."""
    return rng.uniform(0.25, 1, shape) * rng.choice([-1.0, 1.0], shape)


def check(got, ref):
    """got, ref: channels x outputs, float64."""
    err = np.linalg.norm(got - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert err.max() <= 8e-7, err.max()


LAYER_CASES = ["one channel 1e8", "one channel 1e12", "one channel 1e30", "one weight 1e9", "one weight 1e25", "both",
               "units", "huge", "tiny"]


def layer_case(rng, case, C, k):
    x, w = uniform(rng, C, 20, 37), 0.1 * uniform(rng, C, C, k, k)
    if case.startswith("one channel") or case == "both":  # channel 5, as far as the weights are concerned not there
        x[5] *= float(case.split()[-1]) if case != "both" else 1e12
        w[:, 5] = 0
    if case.startswith("one weight") or case == "both":  # a weight that only meets zeros
        w[:, 9] *= float(case.split()[-1]) if case != "both" else 1e12
        x[9] = 0
    if case == "units":  # every channel in a unit of its own, which its weights take back
        unit = 10.0 ** rng.uniform(-12, 12, C)
        x, w = x * unit[:, None, None], w / unit[None, :, None, None]
    if case == "huge":
        x, w = x * 2e37, w * 1e-3
    if case == "tiny":
        x = x * 1e-30
    return x.astype(np.float32), w.astype(np.float32)


@pytest.mark.parametrize("case", LAYER_CASES)
@pytest.mark.parametrize("C,k", [(100, 3), (100, 2), (64, 3)])
def test_layer(handle, C, k, case):
    x, w = layer_case(np.random.default_rng(C + k), case, C, k)
    hwc = torch.zeros((*x.shape[1:], capi.feature_stride(C)), device="cuda")
    hwc[:, :, :C] = torch.as_tensor(x, device="cuda").permute(1, 2, 0)
    y = ops.ConvLayer(handle, w, None, "fp32", act=False)(handle, hwc)
    ref = F.conv2d(torch.as_tensor(x).double()[None], torch.as_tensor(w).double().flip(2, 3))[0].numpy()
    check(y[:, :, :C].permute(2, 0, 1).double().cpu().numpy().reshape(C, -1), ref.reshape(C, -1))


@pytest.mark.parametrize("C,k", [(100, 3), (100, 2), (64, 3)])
def test_layer_of_values_apart(handle, C, k):
    """Values of any sizes side by side, weights of one size: every output pixel is
    off by a share of its own size."""
    rng = np.random.default_rng(2 * C + k)
    x = (uniform(rng, C, 20, 37) * 10.0 ** rng.uniform(-20, 10, (C, 20, 37))).astype(np.float32)
    w = uniform(rng, C, C, k, k).astype(np.float32)
    hwc = torch.zeros((20, 37, capi.feature_stride(C)), device="cuda")
    hwc[:, :, :C] = torch.as_tensor(x, device="cuda").permute(1, 2, 0)
    y = ops.ConvLayer(handle, w, None, "fp32", act=False)(handle, hwc)[:, :, :C].double().cpu().numpy().reshape(-1, C)
    ref = F.conv2d(torch.as_tensor(x).double()[None], torch.as_tensor(w).double().flip(2, 3))[0].numpy()
    check(y, ref.reshape(C, -1).T)


def test_layer_pixels_apart(handle):
    """A pixel out of range takes its tile to float32 products and leaves the other
    tiles' outputs as they are, to the bit."""
    rng = np.random.default_rng(0)
    x, w = layer_case(rng, "", 100, 3)
    w[3, 4] = 0
    layer = ops.ConvLayer(handle, w, None, "fp32")
    hwc = torch.zeros((20, 37, 104), device="cuda")
    hwc[:, :, :100] = torch.as_tensor(x, device="cuda").permute(1, 2, 0)
    want = layer(handle, hwc)
    hwc[2, 3, 7] = 1e-30
    got = layer(handle, hwc)
    assert torch.equal(got[8:], want[8:]) and torch.equal(got[:, 16:], want[:, 16:])


DW_CASES = ["one pixel 1e8", "one pixel 1e12", "one dz 1e9", "both", "columns", "huge", "tiny"]


@pytest.mark.parametrize("case", DW_CASES)
@pytest.mark.parametrize("k", [3, 2])
def test_weight_gradient(handle, case, k):
    """Pixels of one segment: a large one of the input meets a zero of dz and the reverse."""
    rng = np.random.default_rng(k)
    C, H, W = 100, 12, 70
    Ho, Wo = H - k + 1, W - k + 1
    x, dz = uniform(rng, H, W, C), 1e-3 * uniform(rng, Ho, Wo, C)
    if case.startswith("one pixel") or case == "both":
        f = float(case.split()[-1]) if case != "both" else 1e12
        dz[4:4 + k, 8:8 + k] = 0
        x[4 + k - 1, 8 + k - 1] *= f
    if case.startswith("one dz") or case == "both":
        f = float(case.split()[-1]) if case != "both" else 1e12
        x[7:7 + k, 20:20 + k] = 0
        dz[7, 20] *= f
    if case == "columns":  # columns of the map in units of their own, alike products at the first column of taps
        unit = 10.0 ** rng.uniform(-12, 12, (1, W, 1))
        x, dz = x * unit, dz / unit[:, :Wo]
    if case == "huge":
        x, dz = x * 1e30, dz * 1e5
    if case == "tiny":
        x, dz = x * 1e-12, dz * 1e-12
    maps = []
    for m in (x, dz):
        t = torch.zeros((*m.shape[:2], 104), device="cuda")
        t[:, :, :C] = torch.as_tensor(m, device="cuda")
        maps.append(t)
    w = torch.zeros((C, C, k, k), device="cuda")
    _, dw, _ = ops.conv2d_backward_stored(handle, maps[0], torch.zeros_like(maps[1]), w, maps[1], act=False)
    xd, zd = (m[:, :, :C].double().cpu() for m in maps)
    ref = torch.stack([zd.reshape(-1, C).t() @ xd[k - 1 - a:k - 1 - a + Ho, k - 1 - b:k - 1 - b + Wo].reshape(-1, C)
                       for a in range(k) for b in range(k)], dim=2).numpy()
    per_tap = lambda v: v.transpose(0, 2, 3, 1).reshape(-1, C)  # noqa: E731
    check(per_tap(dw.double().cpu().numpy()), per_tap(ref.reshape(C, C, k, k)))


CORR_CASES = ["one channel 1e8", "one channel 1e12", "one channel 1e30", "other map 1e9", "both", "units", "huge",
              "tiny"]


@pytest.mark.parametrize("case", CORR_CASES)
@pytest.mark.parametrize("C,D", [(100, 32), (100, 128), (64, 64), (36, 200)])
def test_correlation(handle, case, C, D):
    rng = np.random.default_rng(C + D)
    H, W = 2, 300
    f0, f1 = uniform(rng, H, W, C), uniform(rng, H, W, C)
    if case.startswith("one channel") or case == "both":
        f0[:, :, 5] *= float(case.split()[-1]) if case != "both" else 1e12
        f1[:, :, 5] = 0
    if case.startswith("other map") or case == "both":
        f1[:, :, 9] *= float(case.split()[-1]) if case != "both" else 1e12
        f0[:, :, 9] = 0
    if case == "units":
        unit = 10.0 ** rng.uniform(-12, 12, C)
        f0, f1 = f0 * unit, f1 / unit
    if case == "huge":
        f0, f1 = f0 * 1e26, f1 * 1e10
    if case == "tiny":
        f0, f1 = f0 * 1e-14, f1 * 1e-14
    maps = []
    for f in (f0, f1):
        t = torch.zeros((H, W, capi.feature_stride(C)), device="cuda")
        t[:, :, :C] = torch.as_tensor(f, device="cuda")
        maps.append(t)
    got = ops.correlation_volume(handle, maps[0], maps[1], C, 0, 1, D, epilogue="raw").double().cpu().numpy()
    a, b = (m[:, :, :C].double().cpu().numpy() for m in maps)
    ref = np.zeros((H, W, D))
    for d in range(D):
        ref[:, d:, d] = (a[:, d:] * b[:, :W - d]).sum(-1)
    check(got.reshape(-1, D).T, ref.reshape(-1, D).T)


def test_correlation_of_values_apart(handle):
    """Values of any sizes in one map, of one size in the other."""
    rng = np.random.default_rng(8)
    f0 = torch.as_tensor(uniform(rng, 2, 300, 104) * 10.0 ** rng.uniform(-20, 10, (2, 300, 104)), dtype=torch.float32)
    f1 = torch.as_tensor(uniform(rng, 2, 300, 104), dtype=torch.float32)
    got = ops.correlation_volume(handle, f0.cuda(), f1.cuda(), 104, 0, 1, 64, epilogue="raw").double().cpu().numpy()
    a, b = f0.double().numpy(), f1.double().numpy()
    ref = np.stack([(a[:, 63:] * b[:, 63 - d:300 - d]).sum(-1) for d in range(64)], axis=-1)
    check(got[:, 63:].reshape(-1, 64), ref.reshape(-1, 64))  # every pixel off by a share of its own size
