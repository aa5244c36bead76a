"""Results in the place of operands that only their own workgroup still reads: O over Q in the fp32 forward, dK over K and dV over V in the
backward.  Bit for bit what separate buffers give, on ordinary rows and on rows that the workgroups redo on the fp32 instruction."""
import numpy as np
import pytest

from autorust_amd import synth
from autorust_amd.device import F32
from gpu_util import Bufs

pytestmark = pytest.mark.gpu

# B, Hq, Hkv, N, D, causal: 32 rows to a workgroup, 128, 256; sums in two halves; a group of query heads
CASES = [(1, 4, 4, 100, 64, False), (8, 16, 16, 257, 64, True), (2, 8, 8, 600, 64, False), (2, 8, 2, 600, 64, True), (1, 4, 4, 200, 128, False),
         (8, 16, 8, 257, 128, False), (1, 12, 12, 1030, 128, False)]


@pytest.mark.parametrize("spread", [False, True])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_in_place(dev, case, spread):
    B, Hq, Hkv, N, D, causal = case
    q, k, v, do = (synth.normal(s, (B, H, N, D)) for s, H in ((41, Hq), (42, Hkv), (43, Hkv), (44, Hq)))
    if spread:  # neither the rows of V nor those of dO fit a common scale
        for x in (v, do):
            x *= np.float32(2.0) ** np.random.default_rng(6).integers(-40, 41, x.shape[:3] + (1,)).astype(np.float32)
    results = []
    with Bufs(dev) as bufs:
        for in_place in (False, True):
            bq, bk, bv, bo = (bufs.put(x) for x in (q, k, v, do))
            o = bufs.new(q.nbytes, zero=False)
            lse, delta = bufs.new(B * Hq * N * 4), bufs.new(B * Hq * N * 4)
            gq = bufs.new(q.nbytes, zero=False)
            gk, gv = (bk, bv) if in_place else (bufs.new(k.nbytes, zero=False), bufs.new(v.nbytes, zero=False))
            dev.flash_fwd_lse(bq, bk, bv, o, lse, B, Hq, Hkv, N, D, F32, causal=causal)
            dev.flash_bwd(bq, bk, bv, o, lse, bo, gq, gk, gv, delta, B, Hq, Hkv, N, D, causal=causal)
            out = [o.copyout(np.float32, q.shape), gq.copyout(np.float32, q.shape), gk.copyout(np.float32, k.shape), gv.copyout(np.float32, v.shape)]
            if in_place:
                bk, bv = bufs.put(k), bufs.put(v)
                dev.flash_fwd(bq, bk, bv, bq, B, Hq, Hkv, N, D, F32, causal=causal)
                out[0] = bq.copyout(np.float32, q.shape)
            results.append(out)
    for name, a, b in zip(("o", "dq", "dk", "dv"), *results):
        assert np.isfinite(a).all(), name
        # (sums of dK and dV over 16 tiles and more are put aside in the result halfway, which in place they cannot be: other roundings of the
        # same sum)
        if name in ("dk", "dv") and Hq // Hkv * -(-N // 32) >= 16:
            assert np.linalg.norm((a - b).astype(np.float64)) <= 2e-6 * np.linalg.norm(a.astype(np.float64)), name
        else:
            assert a.tobytes() == b.tobytes(), name
