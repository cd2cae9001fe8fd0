"""Sweeps of more chains than the three-wave kernel takes (2 per CU; columns of up to 64
labels 4): the checkpointed schemes, with costs kept and streamed, against stored
messages, bit for bit.

The scheme follows the volume's size, which CCS_CRF_SEG_MIN_BYTES moves; it is read
once per process, so a child process takes the other side.  Lengths lie around the
segments of 12 steps and the register ring of three segments.
"""
import hashlib
import json
import os
import subprocess
import sys

import pytest
import torch

from cnn_crf_stereo_amd import capi, ops

pytestmark = pytest.mark.gpu

SMALL = [(n, D) for n in (1, 2, 12, 13, 14, 24, 26, 36, 37, 38, 61) for D in (32, 64, 66, 128)] + [(40, 5), (40, 100)]
EDGES = [(1030, 600, 8), (1030, 1030, 5), (600, 30, 100), (600, 41, 128), (23, 1100, 64), (30, 600, 128)]
LARGE = [(1030, 300, 128), (280, 1100, 128), (1030, 600, 64)]  # streamed: above 128 MiB


def digest(*tensors):
    h = hashlib.sha256()
    for t in tensors:
        h.update(t.contiguous().cpu().numpy().tobytes())
    return h.hexdigest()


def volume(g, H, W, D):
    cost = -torch.softmax(3 * torch.randn((H, W, D), generator=g, device="cuda"), dim=2)
    return cost, *torch.rand((2, H, W), generator=g, device="cuda")


def sweeps(h, H, W, D, directions):
    g = torch.Generator(device="cuda").manual_seed(H + 7 * W + D)
    cost, wx, wy = volume(g, H, W, D)
    A = cost + 0.1 * torch.randn((H, W, D), generator=g, device="cuda")
    sums = torch.zeros((len(directions), 2), dtype=torch.float64, device="cuda")
    for i, d in enumerate(directions):
        ops.slackprop_sweep(h, cost, A, wx, wy, 0.5, 2.0, 2, d, chain_sum=sums[i, 0:], kept_sum=sums[i, 1:])
    return digest(A, sums)


def edges(h, H, W, D):
    g = torch.Generator(device="cuda").manual_seed(H + W + D)
    cost, p, q = volume(g, H, W, D)
    pw = torch.stack([p + 0.1, q + 0.1, 2 * p + 0.3, 2 * q + 0.2])
    pen, _ = ops.pairwise_penalties(h, pw)
    r = ops.slackprop_pw(h, cost, pen, 2, 2, want_unaries=True)
    out = digest(r["labels"], r["sums"], r["unaries"])
    cost[H // 2, W - 1, D // 2] = float("nan")  # the first row sweep finds it in either scheme
    ops.slackprop_pw(h, cost, pen, 2, 1)
    with pytest.raises(capi.CCSError):
        ops.slackprop_status(h)
    return out


def small(h):
    chains = 4 * torch.cuda.get_device_properties(0).multi_processor_count + 3
    out = {}
    for n, D in SMALL:
        out["rows %d %d" % (n, D)] = sweeps(h, chains, n, D, (3, 0))
        out["columns %d %d" % (n, D)] = sweeps(h, n, chains, D, (1, 1))
    for H, W, D in EDGES:
        out["edges %d %d %d" % (H, W, D)] = edges(h, H, W, D)
    return out


def large(h):
    return {"%d %d %d" % (H, W, D): sweeps(h, H, W, D, (3, 1, 0, 1)) for H, W, D in LARGE}


def in_child(which, threshold):
    code = ("import sys, json; sys.path.insert(0, sys.argv[1]); import conftest; "
            "from cnn_crf_stereo_amd import capi; import test_gpu_crf_many_chains as t; "
            "print(json.dumps(t.%s(capi.Handle())))" % which)
    here = os.path.dirname(os.path.abspath(__file__))
    r = subprocess.run([sys.executable, "-c", code, here], env=dict(os.environ, CCS_CRF_SEG_MIN_BYTES=str(threshold)),
                       cwd=here, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    return json.loads(r.stdout.strip().splitlines()[-1])


def test_checkpointed_equal_stored_messages(handle):
    stored, checkpointed = small(handle), in_child("small", 0)
    assert {k for k in stored if stored[k] != checkpointed[k]} == set()


def test_streamed_equal_stored_messages(handle):
    streamed, stored = large(handle), in_child("large", 1 << 40)
    assert {k for k in stored if stored[k] != streamed[k]} == set()
