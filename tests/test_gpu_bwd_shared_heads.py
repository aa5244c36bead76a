"""The fp32 backward where several query heads share a K/V head: dK/dV on 32 keys per workgroup beside dQ on 128 queries, at remainders of
either, around the end of its range, with masks and key lengths, and in the places of K and V."""
import numpy as np
import pytest

import oracle
from autorust_amd import synth
from autorust_amd.device import F32
from gpu_util import Bufs
from test_gpu_bwd import run_fwd_bwd

pytestmark = pytest.mark.gpu


def _inputs(B, Hq, Hkv, N, D):
    return [synth.normal(s, (B, H, N, D)) for s, H in ((71, Hq), (72, Hkv), (73, Hkv), (74, Hq))]


@pytest.mark.parametrize("case", [  # B, Hq, Hkv, N, D, causal, mask, key lengths
    (2, 16, 4, 129, 64, False, False, None), (3, 24, 6, 161, 64, True, False, [161, 33, 0]), (4, 40, 10, 33, 64, False, False, None),
    (2, 24, 4, 255, 64, True, True, None), (1, 32, 8, 512, 64, False, False, [500]), (1, 32, 8, 513, 64, True, False, None), (8, 32, 8, 16, 64, True, False, None),
    (4, 24, 6, 70, 128, False, False, None), (2, 32, 8, 200, 128, True, False, [200, 7]), (2, 16, 8, 300, 128, False, True, None),
    (1, 32, 8, 385, 128, True, False, None), (3, 16, 2, 36, 128, False, False, None),
], ids=str)
def test_backward(dev, case):
    B, Hq, Hkv, N, D, causal, has_mask, lens = case
    q, k, v, do = _inputs(B, Hq, Hkv, N, D)
    mask = synth.normal(75, (N, N)) if has_mask else None
    kv_len = np.array(lens, np.int32) if lens else None
    want = oracle.attention_backward_f64(q, k, v, do, mask=mask, kv_len=kv_len, causal=causal)
    got = run_fwd_bwd(dev, q, k, v, do, mask=mask, kv_len=kv_len, causal=causal)
    for name, g, w in zip(("o", "lse", "dq", "dk", "dv"), got, want):
        err = np.abs(g - w).max()
        assert err <= 3e-5 * max(1.0, np.abs(w).max()), (name, err)
    again = run_fwd_bwd(dev, q, k, v, do, mask=mask, kv_len=kv_len, causal=causal)
    assert all(a.tobytes() == b.tobytes() for a, b in zip(got, again))


@pytest.mark.parametrize("N,D,causal", [(161, 64, False), (200, 128, True)])
def test_gradients_in_the_places_of_keys_and_values(dev, N, D, causal):
    B, Hq, Hkv = 2, 32, 8
    q, k, v, do = _inputs(B, Hq, Hkv, N, D)
    want = run_fwd_bwd(dev, q, k, v, do, causal=causal)
    with Bufs(dev) as bufs:
        dq_, dk_, dv_, ddo = (bufs.put(x) for x in (q, k, v, do))
        o, lse, gq, delta = bufs.new(q.nbytes), bufs.new(B * Hq * N * 4), bufs.new(q.nbytes, zero=False), bufs.new(B * Hq * N * 4, zero=False)
        dev.flash_fwd_lse(dq_, dk_, dv_, o, lse, B, Hq, Hkv, N, D, F32, causal=causal)
        dev.flash_bwd(dq_, dk_, dv_, o, lse, ddo, gq, dk_, dv_, delta, B, Hq, Hkv, N, D, causal=causal)
        for got, w in zip((gq, dk_, dv_), want[2:]):
            assert got.copyout(np.float32, w.shape).tobytes() == w.tobytes()
