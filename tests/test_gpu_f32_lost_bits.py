"""The fp32 kernels on values that a pair of scaled fp16 values cuts short (below 2^-13 of the largest that the scale goes by) where nothing larger
enters the same sum: single channels of 8 neighbouring ones, keys that few attend to, rows far below the others.  Every row and every
channel of a result is held to itself, against the float64 oracle.

Bounds: TOL as in test_gpu_f32_halves.py, six times what N(0,1) operands show.  A logit of size s is off by some roundings of 2^-24 s, and its
probability by as much: where keys stand apart by g in the logits, rows that are made of the lower ones alone are held to g times 2^-19."""
import numpy as np
import pytest

import oracle
from autorust_amd import synth
from autorust_amd.device import F32
from gpu_util import run_flash
from test_gpu_bwd import run_fwd_bwd

pytestmark = pytest.mark.gpu

TOL = 3e-6
F = np.float32

# B, H, N, D: one row to a tile, a single tile, key tiles dealt out between the waves (head size 64, 128), 128 queries per workgroup, two
# groups of waves on 128, 256 queries
SHAPES = [(1, 2, 17, 64), (1, 2, 32, 64), (1, 2, 33, 64), (1, 4, 300, 64), (16, 16, 97, 64), (1, 16, 800, 64), (8, 16, 257, 64), (1, 2, 33, 128),
          (1, 4, 300, 128), (4, 12, 200, 128), (8, 16, 257, 128)]


def close(got, want, tol, name=""):
    """Rows and channels of heads (0, 0) and (0, 1), each by its own norm."""
    got, want = got[:1, :2].astype(np.float64), np.asarray(want, np.float64)
    assert np.isfinite(got).all(), name
    for axis in (-1, -2):
        err, ref = (np.linalg.norm(x, axis=axis) for x in (got - want, want))
        assert (err <= tol * ref).all(), (name, axis, (err[ref > 0] / ref[ref > 0]).max())


def heads(*xs):
    return [x[:1, :2].astype(np.float64) for x in xs]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("e", [10, 20, 30, 38])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_forward_wide_channels(dev, shape, e, causal):
    """Every eighth channel of V, or of K with Q the other way (which leaves the logits alone), 2^e times the rest."""
    q, k, v = (synth.normal(970 + i, shape) for i in range(3))
    up = np.where(np.arange(shape[3]) % 8 == 0, F(2.0 ** e), F(1))
    for a, b, c in ((q, k, v * up), (q / up, k * up, v), (q * up, k / up, v)):
        close(run_flash(dev, a, b, c, F32, causal=causal), oracle.sdpa_f64(*heads(a, b, c), causal=causal), TOL)


@pytest.mark.parametrize("gap", [14, 20, 28])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_forward_sink(dev, shape, gap):
    """A key that all attend to, `gap` above the others, has a row of V that is zero, or zero in half of the channels: O is made of the others' probabilities."""
    q, k, v = (synth.normal(975 + i, shape) for i in range(3))
    q[..., 0], k[..., 0] = 4, 0
    k[..., 5, 0] = gap / 4 * np.sqrt(shape[3])
    for channels in (slice(None), slice(0, None, 2)):
        w = v.copy()
        w[..., 5, channels] = 0
        close(run_flash(dev, q, k, w, F32), oracle.sdpa_f64(*heads(q, k, w)), TOL + gap * 2.0 ** -19)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_forward_zero_channels(dev, shape):
    """Padding: channels that are zero stay zero, and the others what they are."""
    q, k, v = (synth.normal(980 + i, shape) for i in range(3))
    for x in (q, k, v):
        x[..., 41:] = 0
    got = run_flash(dev, q, k, v, F32)
    close(got, oracle.sdpa_f64(*heads(q, k, v)), TOL)
    assert (got[..., 41:] == 0).all()


def difference_terms(q, k, v, do, mask=None, causal=False):
    """What dQ and dK are sums of before dP and D cancel: P (|dO| . |V| + |D|) scale times |K| and |Q|."""
    q, k, v, do = heads(q, k, v, do)
    s = q @ k.swapaxes(-1, -2) / np.sqrt(q.shape[-1]) + (0 if mask is None else mask.astype(np.float64))
    if causal:
        s = np.where(np.tri(q.shape[2], dtype=bool), s, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    d = np.abs((p @ v * do).sum(-1, keepdims=True))
    t = p * (np.abs(do) @ np.abs(v).swapaxes(-1, -2) + d) / np.sqrt(q.shape[-1])
    return t @ np.abs(k), t.swapaxes(-1, -2) @ np.abs(q), np.zeros_like(v)


def check_backward(dev, q, k, v, do, tol=TOL, mask=None, causal=False, rows=slice(None), only=("dq", "dk", "dv")):
    close_backward(run_fwd_bwd(dev, q, k, v, do, mask=mask, causal=causal)[2:], q, k, v, do, tol, mask, causal, rows, only)


def close_backward(got, q, k, v, do, tol=TOL, mask=None, causal=False, rows=slice(None), only=("dq", "dk", "dv"), axes=(-1, -2)):
    """Rows and channels of dq, dk, dv (of the rows `rows`) by their own norms, and four roundings of 2^-24 of the terms that cancel in them."""
    want = oracle.attention_backward_f64(*heads(q, k, v, do), mask=mask, causal=causal)
    terms = difference_terms(q, k, v, do, mask=mask, causal=causal)
    for name, g, w, t in zip(("dq", "dk", "dv"), got, want[2:], terms):
        if name not in only:
            continue
        g, w, t = g[:1, :2, rows].astype(np.float64), np.asarray(w, np.float64)[:, :, rows], t[:, :, rows]
        assert np.isfinite(g).all(), name
        for axis in axes:
            err, ref, cancel = (np.linalg.norm(x, axis=axis) for x in (g - w, w, t))
            bound = tol * ref + 2.0 ** -22 * cancel
            assert (err <= bound).all(), (name, axis, (err[bound > 0] / bound[bound > 0]).max() * tol)


@pytest.mark.parametrize("which", ["q", "dout"])
@pytest.mark.parametrize("e", [20, 30, 38])
@pytest.mark.parametrize("N, causal", [(9, False), (16, False), (32, False), (129, True), (160, True), (257, True)])
@pytest.mark.parametrize("D", [64, 128])
def test_backward_a_single_tile_of_queries(dev, D, N, causal, e, which):
    """Key blocks that see no second tile of queries (all of N <= 32, the last one of a causal head): channels 8 .. 15 of Q, or of dO, 2^-e of the
    others come out in dK and dV as they should."""
    q, k, v, do = (synth.normal(985 + i, (8, 16, N, D)) for i in range(4))
    (q if which == "q" else do)[..., 8:16] *= F(2.0 ** -e)
    check_backward(dev, q, k, v, do, causal=causal, rows=slice(N - 1 - (N - 1) % 128, None), only=("dk", "dv"))


@pytest.mark.parametrize("how", ["key", "mask", "one key"])
@pytest.mark.parametrize("gap, causal", [(8, False), (14, False), (20, False), (28, False), (20, True)])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_backward_keys_that_few_attend_to(dev, shape, gap, causal, how):
    """Every other key, or a single one, `gap` below the others in the logits, by K or by an additive mask: its rows of dK and dV are made of small probabilities alone."""
    N = shape[2]
    q, k, v, do = (synth.normal(990 + i, shape) for i in range(4))
    mask = None
    if how == "mask":
        mask = np.zeros((N, N), F)
        mask[:, ::2] = -gap
    else:
        q[..., 0], k[..., 0] = 4, 0
        k[..., slice(0, None, 2) if how == "key" else N // 2, 0] = -gap / 4 * np.sqrt(shape[3])
    # (causal: query 0 sees key 0 alone, which all later ones avoid; its difference of dP and D is nothing but roundings)
    check_backward(dev, q, k, v, do, TOL + gap * 2.0 ** -19, mask=mask, causal=causal, rows=slice(1 if causal else 0, None), only=("dk", "dv"))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("e", [14, 20, 28])
@pytest.mark.parametrize("which", ["q", "dout"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_backward_small_rows(dev, shape, which, e, causal):
    """The later half of the rows of Q, or of dO, 2^-e of the earlier: under the causal mask late keys see no others."""
    q, k, v, do = (synth.normal(995 + i, shape) for i in range(4))
    (q if which == "q" else do)[..., shape[2] // 2:, :] *= F(2.0 ** -e)
    check_backward(dev, q, k, v, do, causal=causal)


@pytest.mark.parametrize("e", [10, 14, 20, 30])
@pytest.mark.parametrize("shape, causal", [(s, False) for s in SHAPES] + [(s, True) for s in SHAPES + [(8, 16, 129, 64), (8, 16, 129, 128)]], ids=str)
def test_backward_wide_channels(dev, shape, causal, e):
    """Every eighth channel of an operand 2^e times the rest, with its counterpart in a product the other way or not: the other channels of the results."""
    q, k, v, do = (synth.normal(1000 + i, shape) for i in range(4))
    up = np.where(np.arange(shape[3]) % 8 == 0, F(2.0 ** e), F(1))
    for x in ((q / up, k * up, v, do), (q * up, k / up, v, do), (q, k, v * up, do), (q, k, v, do * up), (q, k, v / up, do * up), (q, k, v * up, do / up)):
        # (causal: query 0 sees one key, its difference of dP and D is nothing but roundings)
        check_backward(dev, *x, causal=causal, rows=slice(1 if causal else 0, None))


@pytest.mark.parametrize("which", ["q", "k", "v", "dout", "all"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_backward_zero_channels(dev, shape, which):
    """Padding: channels that are zero, in all operands or in one; and one row that has them, 2^-30 of the others."""
    x = dict(zip(("q", "k", "v", "dout"), (synth.normal(1010 + i, shape) for i in range(4))))
    for name in x if which == "all" else [which]:
        x[name][..., 41:] = 0
    check_backward(dev, *x.values())
    if which != "all" and shape[2] <= 257:
        x[which][..., 3, 41:] = F(2.0 ** -30)
        check_backward(dev, *x.values())


@pytest.mark.parametrize("gap", [8, 14, 20, 28])
@pytest.mark.parametrize("shape", [(1, 2, 32, 64), (1, 4, 300, 64), (16, 16, 100, 64), (1, 16, 800, 64), (8, 16, 260, 64), (1, 4, 300, 128), (4, 12, 200, 128)], ids=str)
def test_backward_channels_that_few_have(dev, shape, gap):
    """A channel of K, of Q and of dO that is zero wherever keys and queries attend to each other: what dQ, dK and dV have of it is made of probabilities
    `gap` below the others alone."""
    N, half = shape[2], shape[2] // 2
    last = -(-half // 128) * 128  # whole blocks of the later half of the keys
    q, k, v, do = (synth.normal(1020 + i, shape) for i in range(4))
    q[..., 0], k[..., 0] = 4, 0
    k[..., ::2, 0] = -gap / 4 * np.sqrt(shape[3])
    check_backward(dev, q, k, v, do, TOL + gap * 2.0 ** -19, only=("dq",))
    q, k, v, do = (synth.normal(1030 + i, shape) for i in range(4))
    mask = np.zeros((N, N), F)
    mask[:half, half:] = -gap
    q[..., half:, 9] = do[..., half:, 9] = 0
    if last < N:
        check_backward(dev, q, k, v, do, TOL + gap * 2.0 ** -19, mask=mask, rows=slice(last, None), only=("dk", "dv"))


@pytest.mark.parametrize("e", [14, 20, 28])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_backward_small_rows_of_v(dev, shape, e):
    """The earlier half of the rows of V 2^-e of the later: under the causal mask early queries see no others, dP is small, and dQ with it."""
    q, k, v, do = (synth.normal(1040 + i, shape) for i in range(4))
    v[..., : shape[2] // 2, :] *= F(2.0 ** -e)
    check_backward(dev, q, k, v, do, causal=True, rows=slice(1, None))
