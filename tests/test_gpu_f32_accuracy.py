"""Accuracy of the fp32 kernels on N(0,1) operands: relative error (2-norm over sampled heads, against float64).  The bounds are what
v_mfma_f32_32x32x2_f32 gave on these inputs, with the key (query) tiles of these grids dealt out to four sums, and 3 %; a single sum
that is rounded with each of the 12 matrix instructions of a tile gave, forward, 4.9e-7 at N = 789 and 7.7e-7 at N = 2048, and in dV
6.1e-7 and 9.4e-7."""
import numpy as np
import pytest

import oracle
from autorust_amd import host, synth
from autorust_amd.device import F32
from gpu_util import run_flash
from test_gpu_bwd import run_fwd_bwd

pytestmark = pytest.mark.gpu

SEED = 10 ** 6   # (neighbouring seeds give sequences that are shifted against each other, and outputs twice as large)

# B, H, N, D, bounds without and with a mask: 256 queries per workgroup (head size 64, 128), 128 queries, the same with short heads
FORWARD = [(8, 6, 789, 64, 3.94e-7, 3.94e-7), (2, 12, 2048, 128, 5.98e-7, 5.97e-7), (1, 16, 2048, 128, 5.98e-7, 5.97e-7),
           (8, 12, 197, 64, 3.31e-7, 3.04e-7), (8, 12, 197, 128, 4.32e-7, 3.59e-7)]


def _error(got, want):
    got, want = (np.asarray(x, np.float64) for x in (got, want))
    return np.linalg.norm(got - want) / np.linalg.norm(want)


def _sample(B, H):
    return [(0, 0), (B - 1, H - 1)]


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("case", FORWARD, ids=str)
def test_forward(dev, case, masked):
    B, H, N, D = case[:4]
    q, k, v = (synth.normal(970 + SEED * i, (B, H, N, D)) for i in range(3))
    mask = synth.normal(970 + 5 * SEED, (N, N)) if masked else None
    got = run_flash(dev, q, k, v, F32, mask=mask)
    at = _sample(B, H)
    want = [oracle.sdpa_f64(q[b:b + 1, h:h + 1], k[b:b + 1, h:h + 1], v[b:b + 1, h:h + 1], mask=mask)[0, 0] for b, h in at]
    assert _error([got[b, h] for b, h in at], want) <= case[4 + masked]


def test_forward_through_the_tensor_interface():
    B, H, N, D = 8, 6, 789, 64
    q, k, v = (synth.normal(970 + SEED * i, (B, H, N, D)) for i in range(3))
    hdev = host.HipDevice(0)
    tq, tk, tv = (host.Tensor.from_slice(hdev, x, x.shape) for x in (q, k, v))
    got = tq.flash_attention_with(tk, tv, None, 0.0, False, host.Session()).to_list()
    at = _sample(B, H)
    want = [oracle.sdpa_f64(q[b:b + 1, h:h + 1], k[b:b + 1, h:h + 1], v[b:b + 1, h:h + 1])[0, 0] for b, h in at]
    assert _error([got[b, h] for b, h in at], want) <= FORWARD[0][4]


# B, H, N, D, causal, bounds of dq, dk, dv: dQ and dK/dV apart (head size 64), in one grid (128; causal on a short one: 64)
BACKWARD = [(8, 6, 789, 64, False, 5.91e-7, 5.88e-7, 5.69e-7), (4, 8, 512, 64, False, 5.55e-7, 5.58e-7, 5.34e-7),
            (1, 16, 2048, 128, False, 8.22e-7, 8.18e-7, 8.11e-7), (1, 4, 512, 128, False, 6.60e-7, 6.59e-7, 6.28e-7),
            (4, 8, 512, 64, True, 4.22e-7, 4.77e-7, 4.21e-7), (1, 4, 4096, 128, True, 5.96e-7, 9.33e-7, 9.01e-7)]


@pytest.mark.parametrize("case", BACKWARD, ids=str)
def test_backward(dev, case):
    B, H, N, D, causal = case[:5]
    q, k, v, do = (synth.normal(980 + SEED * i, (B, H, N, D)) for i in range(4))
    got = run_fwd_bwd(dev, q, k, v, do, causal=causal)
    at = _sample(B, H) if N < 4096 else [(0, 0)]
    want = [oracle.attention_backward_f64(*(x[b:b + 1, h:h + 1] for x in (q, k, v, do)), causal=causal) for b, h in at]
    for i, name in ((2, "dq"), (3, "dk"), (4, "dv")):
        assert _error([got[i][b, h] for b, h in at], [w[i][0, 0] for w in want]) <= case[3 + i], name
