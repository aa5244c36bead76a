"""The fp32 forward where several groups of waves share the keys of the same queries and turn their rows around in LDS: heads of so few keys
that some groups have none, the last rows of a head past the end; against the float64 oracle, and the same bits on every pass."""
import numpy as np
import pytest

import oracle
from autorust_amd import synth
from autorust_amd.device import F32
from gpu_util import Bufs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal,masked", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("B,H,N,D", [(1, 3, 1, 64), (1, 24, 36, 64), (2, 6, 127, 128), (4, 8, 734, 64), (1, 4, 1000, 128)])
def test_forward(dev, B, H, N, D, causal, masked):
    q, k, v = (synth.normal(s, (B, H, N, D)) for s in (31, 32, 33))
    mask = synth.normal(34, (N, N)) if masked else None
    with Bufs(dev) as bufs:
        dq, dk, dv, dm = (bufs.put(x) if x is not None else None for x in (q, k, v, mask))
        outs = []
        for _ in range(6):
            o, lse = bufs.new(q.nbytes, zero=False), bufs.new(B * H * N * 4, zero=False)
            dev.flash_fwd_lse(dq, dk, dv, o, lse, B, H, H, N, D, F32, mask=dm, causal=causal)
            outs.append((o.copyout(np.float32, q.shape), lse.copyout(np.float32, q.shape[:3])))
    # 2^-19 of the largest |V| of the head: |P error| is some 2^-20 of P (a logit of up to 8 carries 2^-21 of itself and the exponential a unit)
    bound = 2.0 ** -19 * np.abs(v).max(axis=(2, 3))[:, :, None, None]
    assert (np.abs(outs[0][0] - oracle.sdpa_f64(q, k, v, mask=mask, causal=causal)) <= bound).all()
    assert np.abs(outs[0][1] - oracle.lse_f64(q, k, mask=mask, causal=causal)).max() <= 4e-6
    assert all(x.tobytes() == y.tobytes() for out in outs[1:] for x, y in zip(out, outs[0]))
