"""Accuracy of the fp32 kernels: relative error (2-norm over sampled heads, against float64).  The bounds are what
v_mfma_f32_32x32x2_f32 gave on these inputs, with the key tiles of these grids dealt out to four sums, and 3 %; a single sum that is
rounded with each of the 12 matrix instructions of a tile gave 3.8e-7 at N = 789 and 5.8e-7 at N = 2048."""
import numpy as np
import pytest

import oracle
from autorust_amd import host, synth
from autorust_amd.device import F32
from gpu_util import run_flash

pytestmark = pytest.mark.gpu

# B, H, N, D, bounds without and with a mask: 256 queries per workgroup (head size 64, 128), 128 queries, the same with short heads
FORWARD = [(8, 6, 789, 64, 2.12e-7, 2.68e-7), (2, 12, 2048, 128, 2.88e-7, 3.70e-7), (1, 16, 2048, 128, 2.88e-7, 3.70e-7),
           (8, 12, 197, 64, 2.63e-7, 2.80e-7), (8, 12, 197, 128, 3.30e-7, 3.41e-7)]


def _error(got, want):
    got, want = (np.asarray(x, np.float64) for x in (got, want))
    return np.linalg.norm(got - want) / np.linalg.norm(want)


def _sample(B, H):
    return [(0, 0), (B - 1, H - 1)]


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("case", FORWARD, ids=str)
def test_forward(dev, case, masked):
    B, H, N, D = case[:4]
    q, k, v = (synth.normal(970 + i, (B, H, N, D)) for i in range(3))
    mask = synth.normal(975, (N, N)) if masked else None
    got = run_flash(dev, q, k, v, F32, mask=mask)
    at = _sample(B, H)
    want = [oracle.sdpa_f64(q[b:b + 1, h:h + 1], k[b:b + 1, h:h + 1], v[b:b + 1, h:h + 1], mask=mask)[0, 0] for b, h in at]
    assert _error([got[b, h] for b, h in at], want) <= case[4 + masked]


def test_forward_through_the_tensor_interface():
    B, H, N, D = 8, 6, 789, 64
    q, k, v = (synth.normal(970 + i, (B, H, N, D)) for i in range(3))
    hdev = host.HipDevice(0)
    tq, tk, tv = (host.Tensor.from_slice(hdev, x, x.shape) for x in (q, k, v))
    got = tq.flash_attention_with(tk, tv, None, 0.0, False, host.Session()).to_list()
    at = _sample(B, H)
    want = [oracle.sdpa_f64(q[b:b + 1, h:h + 1], k[b:b + 1, h:h + 1], v[b:b + 1, h:h + 1])[0, 0] for b, h in at]
    assert _error([got[b, h] for b, h in at], want) <= FORWARD[0][4]
