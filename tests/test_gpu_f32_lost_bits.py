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
