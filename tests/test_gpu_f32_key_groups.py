"""The fp32 forward with two groups of 4 waves on 128 queries, which deal the key tiles out between them: sizes and key lengths at which a
group has no tile, one, or one more than the other."""
import numpy as np
import pytest

import oracle
from autorust_amd import synth
from autorust_amd.device import F32
from gpu_util import Bufs

pytestmark = pytest.mark.gpu

# B, Hq, Hkv, N, causal, mask, key lengths; few enough workgroups to run at once, too many of 32 queries
CASES = [
    (6, 8, 8, 512, False, False, [0, 1, 32, 33, 64, 512]), (3, 16, 4, 545, False, False, None), (6, 8, 8, 513, True, False, [513, 1, 31, 65, 96, 97]),
    (2, 24, 24, 570, True, True, None), (4, 12, 12, 601, False, True, [601, 40, 577, 576]), (1, 16, 16, 1503, False, False, None),
    (1, 16, 8, 1504, True, False, None),
]


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_forward(dev, case, wide):
    B, Hq, Hkv, N, causal, has_mask, lens = case
    D = 64
    q, k, v = (synth.normal(s, (B, H, N, D)) for s, H in ((31, Hq), (32, Hkv), (33, Hkv)))
    if wide:  # rows and channels that no common scale fits: the workgroups redo them in fp32
        rng = np.random.default_rng(5)
        v = v * np.float32(2.0) ** rng.integers(-30, 31, (B, Hkv, N, 1)).astype(np.float32)
        v = v * np.float32(2.0) ** rng.integers(-15, 16, (B, Hkv, 1, D)).astype(np.float32)
    mask = synth.normal(34, (N, N)) if has_mask else None
    kv_len = np.array(lens, np.int32) if lens else None
    with Bufs(dev) as bufs:
        dq, dk, dv = (bufs.put(x) for x in (q, k, v))
        o, lse = bufs.new(q.nbytes, zero=False), bufs.new(B * Hq * N * 4, zero=False)
        dm = bufs.put(mask) if has_mask else None
        dl = bufs.put(kv_len) if lens else None
        dev.flash_fwd_lse(dq, dk, dv, o, lse, B, Hq, Hkv, N, D, F32, mask=dm, kv_len=dl, causal=causal)
        got, got_lse = o.copyout(np.float32, q.shape), lse.copyout(np.float32, q.shape[:3])
    want = oracle.sdpa_f64(q, k, v, mask=mask, kv_len=kv_len, causal=causal)
    if lens:
        want[kv_len == 0] = 0.0  # no key: zeros, not a softmax of nothing
    want_lse = oracle.lse_f64(q, k, mask=mask, kv_len=kv_len, causal=causal)
    # |P error| is some 2^-20 of P (a logit of up to 8 carries 2^-21 of itself and the exponential a unit): 2^-19 of the largest |V| of the head
    bound = 2.0 ** -19 * np.abs(v).max(axis=(2, 3)).repeat(Hq // Hkv, axis=1)[:, :, None, None]
    if wide:  # ... and of what the row sees in the channel
        bound = 2.0 ** -19 * oracle.sdpa_f64(q, k, np.abs(v), mask=mask, kv_len=kv_len, causal=causal)
        if lens:
            bound[kv_len == 0] = 0.0
    assert (np.abs(got - want) <= bound).all()
    seen = np.isfinite(want_lse) & (want_lse > -1e29)
    assert np.abs(got_lse - want_lse)[seen].max() <= 4e-6 and (got_lse[~seen] < -1e29).all()
