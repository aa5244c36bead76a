"""The fp32 forward on four waves to 32 queries, on either side of the lengths at which own rows are read whole or by the lanes that own them:
against the float64 oracle, and the same bits on every pass."""
import numpy as np
import pytest

import oracle
from autorust_amd import synth
from autorust_amd.device import F32
from gpu_util import Bufs

pytestmark = pytest.mark.gpu

EDGES = [(64, False, N) for N in (160, 161, 288, 289)] + [(64, True, N) for N in (128, 129, 152, 153, 528, 529, 767, 768)] + \
        [(128, False, N) for N in (32, 33, 64, 65, 999)] + [(128, True, N) for N in (84, 85, 266, 267, 512)]


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("D,causal,N", EDGES)
def test_forward(dev, D, causal, N, masked):
    B, H = 1, 4
    q, k, v = (synth.normal(s, (B, H, N, D)) for s in (51, 52, 53))
    mask = synth.normal(54, (N, N)) if masked else None
    with Bufs(dev) as bufs:
        dq, dk, dv, dm = (bufs.put(x) if x is not None else None for x in (q, k, v, mask))
        outs = []
        for _ in range(3):
            o, lse = bufs.new(q.nbytes, zero=False), bufs.new(B * H * N * 4, zero=False)
            dev.flash_fwd_lse(dq, dk, dv, o, lse, B, H, H, N, D, F32, mask=dm, causal=causal)
            outs.append((o.copyout(np.float32, q.shape), lse.copyout(np.float32, q.shape[:3])))
    # 2^-19 of the largest |V| of the head: |P error| is some 2^-20 of P (a logit of up to 8 carries 2^-21 of itself and the exponential a unit)
    bound = 2.0 ** -19 * np.abs(v).max(axis=(2, 3))[:, :, None, None]
    assert (np.abs(outs[0][0] - oracle.sdpa_f64(q, k, v, mask=mask, causal=causal)) <= bound).all()
    assert np.abs(outs[0][1] - oracle.lse_f64(q, k, mask=mask, causal=causal)).max() <= 4e-6
    assert all(x.tobytes() == y.tobytes() for out in outs[1:] for x, y in zip(out, outs[0]))
