"""The fp32 backward on grids of more than two and at most three workgroups per compute unit, where the waves of dQ go first, and beside
their ends: against the float64 oracle, and the same bits every time."""
import numpy as np
import pytest

import oracle
from autorust_amd import synth
from test_gpu_bwd import run_fwd_bwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [85, 86, 128, 129])  # 510, 516, 768 and 774 workgroups
def test_backward(dev, H):
    q, k, v, do = (synth.normal(s, (1, H, 290, 64)) for s in (31, 32, 33, 34))
    want = oracle.attention_backward_f64(q, k, v, do)
    got = run_fwd_bwd(dev, q, k, v, do)
    for name, g, w in zip(("o", "lse", "dq", "dk", "dv"), got, want):
        err = np.abs(g - w).max()
        assert err <= 3e-5 * max(1.0, np.abs(w).max()), (name, err)
    again = run_fwd_bwd(dev, q, k, v, do)
    assert all(a.tobytes() == b.tobytes() for a, b in zip(got, again))
