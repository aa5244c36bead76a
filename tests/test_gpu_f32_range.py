"""The fp32 kernels on operands that are not the exact sum of three bf16 values: infinities, values that round to infinity in bf16
and values below 2^-110.  Such workgroups compute on the fp32 matrix instruction; what they give is held to the float64 oracle as
ordinary data is, in every tiling."""
import numpy as np
import pytest

import oracle
from autorust_amd import synth
from autorust_amd.device import F32
from gpu_util import run_flash
from test_gpu_bwd import run_fwd_bwd

pytestmark = pytest.mark.gpu

HUGE = np.float32(3.4e38)    # rounds to infinity in bf16
# B, H, N, D: key tiles dealt out between the waves (head size 64, 128), 128 queries per workgroup, 256 queries
SHAPES = [(1, 2, 70, 64), (1, 2, 70, 128), (16, 16, 97, 64), (16, 16, 65, 128), (8, 16, 257, 64), (8, 16, 257, 128)]
J = 5                        # the key (or query) that holds the value, in channel 7 of head (0, 0); head (0, 1) is left alone
EDGE = (0, 0, J, 7)


def _qkv(shape):
    B, H, N, D = shape
    return [synth.normal(950 + i, (B, H, N, D)) for i in range(3)]


def _heads(x):
    return x[:1, :2].astype(np.float64)


def _close(got, want, tol=4e-6):
    """Elementwise against the largest value of the row's head; the same values where the result is not finite."""
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[~fin], want[~fin].astype(np.float32), equal_nan=True)
    assert np.abs(got[fin] - want[fin]).max() <= tol * max(1.0, np.abs(want[fin]).max())


@pytest.mark.parametrize("form", ["plain", "causal", "mask"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_forward(dev, shape, form):
    B, H, N, D = shape
    causal = form == "causal"
    mask = synth.normal(960, (N, N)) if form == "mask" else None

    def check(q, k, v, want_kv=None):
        got = run_flash(dev, q, k, v, F32, mask=mask, causal=causal)[:1, :2]
        kk, vv = want_kv or (k, v)
        want = oracle.sdpa_f64(_heads(q), _heads(kk), _heads(vv), mask=mask, causal=causal)
        for h in range(2):
            _close(got[0, h], want[0, h])

    q, k, v = _qkv(shape)
    big = v.copy()
    big[EDGE] = HUGE
    got = run_flash(dev, q, k, big, F32, mask=mask, causal=causal)[0, :2]
    want = oracle.sdpa_f64(_heads(q), _heads(k), _heads(big), mask=mask, causal=causal)[0]
    assert np.isfinite(got).all()
    chan = np.arange(D) == 7
    _close(got[0][:, ~chan], want[0][:, ~chan])
    _close(got[0][:, chan], want[0][:, chan])
    _close(got[1], want[1])

    inf = v.copy()
    inf[EDGE] = np.inf
    got = run_flash(dev, q, k, inf, F32, mask=mask, causal=causal)[0, :2]
    seen = slice(32, None)                    # (rows of the causal diagonal tile multiply the key by a probability of zero)
    assert (got[0, seen, 7] == np.inf).all()
    want = oracle.sdpa_f64(_heads(q), _heads(k), _heads(v), mask=mask, causal=causal)[0]
    _close(got[0][:, ~chan], want[0][:, ~chan])
    _close(got[1], want[1])

    # a key whose logit is -inf drops out; one whose huge channel meets zeros does not count in it
    qp = q.copy()
    qp[0, 0, :, 7] = np.abs(qp[0, 0, :, 7]) + np.float32(0.1)
    kd = k.copy()
    kd[EDGE] = -np.inf
    drop = k.copy()
    drop[EDGE] = -1e30                        # finite in float64: a probability of exactly zero there
    check(qp, kd, v, want_kv=(drop, v))
    qz = q.copy()
    qz[0, 0, :, 7] = 0
    kz = k.copy()
    kz[EDGE] = HUGE
    check(qz, kz, v)

    # a query that is not a number spoils its own row
    qn = q.copy()
    qn[EDGE] = np.nan
    got = run_flash(dev, qn, k, v, F32, mask=mask, causal=causal)[0, :2]
    want = oracle.sdpa_f64(_heads(q), _heads(k), _heads(v), mask=mask, causal=causal)[0]
    assert np.isnan(got[0, J]).all()
    rest = np.arange(N) != J
    _close(got[0][rest], want[0][rest])
    _close(got[1], want[1])


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_forward_small_values(dev, shape):
    """Powers of two taken out of V, and moved from K to Q, leave the relative accuracy alone (fp32 products do not lose bits above
    2^-126; 2^-116 is below what three bf16 values hold)."""
    q, k, v = _qkv(shape)
    tiny = np.float32(2.0 ** -116)
    want = oracle.sdpa_f64(_heads(q), _heads(k), _heads(v))
    got = run_flash(dev, q, k, v * tiny, F32)[:1, :2].astype(np.float64) * 2.0 ** 116
    assert np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want)
    got = run_flash(dev, q / tiny, k * tiny, v, F32)[:1, :2]
    assert np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want)
    got = run_flash(dev, q * tiny, k / tiny, v, F32)[:1, :2]
    assert np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want)
    # one small value among ordinary ones
    one = v.copy()
    one[EDGE] = np.float32(1e-38)
    got = run_flash(dev, q, k, one, F32)[:1, :2]
    want = oracle.sdpa_f64(_heads(q), _heads(k), _heads(one))
    assert np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_backward(dev, shape, causal):
    B, H, N, D = shape
    q, k, v = _qkv(shape)
    do = synth.normal(955, shape)

    def check(q, k, v, do, scale_out=1.0):
        got = run_fwd_bwd(dev, q, k, v, do, causal=causal)
        want = oracle.attention_backward_f64(_heads(q), _heads(k), _heads(v), _heads(do), causal=causal)
        for name, g, w in zip(("o", "lse", "dq", "dk", "dv"), got, want):
            g = g[:1, :2].astype(np.float64)
            assert np.isfinite(g).all(), name
            for h in range(2):
                # channel by channel, so that a huge one does not hide the others
                gg, ww = (x[0, h].reshape(N, -1).astype(np.float64) for x in (g, w))
                err, ref = np.linalg.norm(gg - ww, axis=0), np.linalg.norm(ww, axis=0)
                assert (err <= 5e-6 * np.maximum(ref, 1e-3 * np.median(ref))).all(), (name, h, (err / ref).max())

    # a huge gradient in a channel where V is zero: dV is huge and finite, everything else as ever
    vz, big = v.copy(), do.copy()
    vz[0, 0, :, 7] = 0
    big[EDGE] = HUGE
    check(q, k, vz, big)
    # a huge K in a channel where Q is zero: dQ is huge and finite there
    qz, kz = q.copy(), k.copy()
    qz[0, 0, :, 7] = 0
    kz[EDGE] = HUGE * np.float32(0.999)
    check(qz, kz, v, do * np.float32(1e-3))
    # gradients and values below what three bf16 values hold
    tiny = np.float32(2.0 ** -100)
    check(q, k, v, do * tiny)
    check(q, k, v * tiny, do)
