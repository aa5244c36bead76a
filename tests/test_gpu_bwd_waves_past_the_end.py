"""The fp32 backward where the last workgroup of a head has waves without rows: they say nothing about the bits that its operands have lost.
A power of two from Q to K changes neither the logits nor the bits of anything that is scaled by its own largest value, so the
gradients are those of the unscaled operands times that power, bit for bit, unless a workgroup falls back to the fp32 instruction."""
import numpy as np
import pytest

from autorust_amd import synth
from autorust_amd.device import F32
from gpu_util import Bufs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("up", [13, -13])
@pytest.mark.parametrize("case", [  # B, Hq, Hkv, N, D, causal
    (4, 16, 16, 197, 64, False), (4, 16, 16, 197, 64, True), (1, 64, 64, 129, 64, False), (2, 32, 32, 224, 64, False), (2, 48, 48, 545, 64, False),
    (4, 12, 12, 20, 64, False), (2, 16, 4, 161, 64, False), (2, 32, 32, 256, 64, False), (2, 32, 32, 197, 128, False),
], ids=str)
def test_backward_of_reciprocal_scales(dev, case, up):
    B, Hq, Hkv, N, D, causal = case
    q, k, v, do = (synth.normal(s, (B, H, N, D)) for s, H in ((81, Hq), (82, Hkv), (83, Hkv), (84, Hq)))
    lse_shape = (B, Hq, N)
    with Bufs(dev) as bufs:
        dv_, ddo, o, lse = bufs.put(v), bufs.put(do), bufs.new(q.nbytes), bufs.new(B * Hq * N * 4)
        dev.flash_fwd_lse(bufs.put(q), bufs.put(k), dv_, o, lse, B, Hq, Hkv, N, D, F32, causal=causal)
        assert np.isfinite(lse.copyout(np.float32, lse_shape)).all()

        def grads(e):
            gq, gk, gv, delta = bufs.new(q.nbytes, zero=False), bufs.new(k.nbytes, zero=False), bufs.new(v.nbytes, zero=False), bufs.new(B * Hq * N * 4)
            dev.flash_bwd(bufs.put(np.ldexp(q, -e)), bufs.put(np.ldexp(k, e)), dv_, o, lse, ddo, gq, gk, gv, delta, B, Hq, Hkv, N, D, causal=causal)
            return [np.ldexp(g.copyout(np.float32, x.shape), s) for g, x, s in ((gq, q, -e), (gk, k, e), (gv, v, 0))]

        for name, a, b in zip(("dq", "dk", "dv"), grads(0), grads(up)):
            rows = np.unique(np.nonzero((a != b).any(axis=3))[2])
            assert rows.size == 0, (name, rows)
