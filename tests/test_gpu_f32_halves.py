"""The fp32 kernels on operands whose values are far apart: fp32 operands are taken as two fp16 values each, scaled by the largest value
of a row or of a stream of tiles, so these are the inputs on which a scale can be wrong.  Every tiling, against the float64 oracle.
(Values that lose bits with nothing larger beside them, in single channels and rows: test_gpu_f32_lost_bits.py.)

Bounds: a product of such operands is off by at most 2^-22 of itself and a sum of them by a few roundings of 2^-24, as long as the
values that matter are within the window of the scale; outside of it the kernels take the fp32 matrix instruction.  Either way errors
stay below 3e-6 of the row (outputs) or of the channel (gradients), six times what N(0,1) operands show here."""
import numpy as np
import pytest

import oracle
from autorust_amd import synth
from autorust_amd.device import F32
from gpu_util import run_flash
from test_gpu_bwd import run_fwd_bwd
from test_gpu_f32_lost_bits import close_backward

pytestmark = pytest.mark.gpu

# B, H, N, D: key tiles dealt out between the waves (head size 64, 128), 128 queries per workgroup, 256 queries
SHAPES = [(1, 2, 70, 64), (1, 2, 70, 128), (16, 16, 97, 64), (4, 12, 200, 128), (8, 16, 257, 64), (8, 16, 257, 128)]
TOL = 3e-6


def _inputs(shape, kind):
    q, k, v, do = (synth.normal(990 + 10 ** 6 * i, shape) for i in range(4))
    f = lambda e: np.float32(2.0 ** e)
    N = shape[2]
    if kind == "small channels":             # in every operand, 2^-20 of the others
        for x in (k, v, do):
            x[..., 8:16] *= f(-20)
        q[..., 8:16] *= f(-18)
    elif kind == "channels against each other":   # as much of every logit comes from either half of the channels; within the window
        q[..., : shape[3] // 2] *= f(9)
        k[..., : shape[3] // 2] *= f(-9)
    elif kind == "growing":                  # later rows 2^10 times the first tile's
        v[..., 40:, :] *= f(10)
        do[..., : N - 40, :] *= f(10)
    elif kind == "zeros first":
        k[..., :32, :] = 0
        v[..., :33, :] = 0
        do[..., N - 32:, :] = 0
        do *= f(-20)
    elif kind == "ranges":                   # of whole tensors
        q *= f(60)
        k *= f(-60)
        v *= f(-40)
        do *= f(70)
    elif kind == "small rows that count":    # every query attends to rows of V that are 2^-16 of the others
        q[..., 0] = 3
        k[..., 0] = 0
        k[..., N // 2:, 0] = 6 * np.sqrt(shape[3])   # logits of 18: probabilities are off by some 6 roundings of 2^-20
        v[..., N // 2:, :] *= f(-16)
    return q, k, v, do


KINDS = ["small channels", "channels against each other", "growing", "zeros first", "ranges"]


@pytest.mark.parametrize("kind", KINDS + ["small rows that count"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_forward(dev, shape, kind):
    q, k, v, _ = _inputs(shape, kind)
    got = run_flash(dev, q, k, v, F32)[:1, :2].astype(np.float64)
    want = oracle.sdpa_f64(q[:1, :2], k[:1, :2], v[:1, :2])
    tol = 2e-5 if kind == "small rows that count" else TOL
    for axis in (-1, -2):                    # by rows, and by channels
        assert (np.linalg.norm(got - want, axis=axis) <= tol * np.linalg.norm(want, axis=axis)).all()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_backward(dev, shape, kind, causal):
    q, k, v, do = _inputs(shape, kind)
    got = run_fwd_bwd(dev, q, k, v, do, causal=causal)
    want = oracle.attention_backward_f64(*(x[:1, :2].astype(np.float64) for x in (q, k, v, do)), causal=causal)
    for name, g, w in zip(("dq", "dk", "dv"), got[2:], want[2:]):
        err = np.linalg.norm(g[:1, :2].astype(np.float64) - w, axis=-2)
        ref = np.linalg.norm(w.astype(np.float64), axis=-2)
        # (a channel that cancels almost to nothing is held to the others)
        assert (err <= TOL * np.maximum(ref, 2.0 ** -21 * ref.max(axis=-1, keepdims=True))).all(), (name, (err / ref).max())
    # and by rows.  (Causal: query 0 sees one key, its difference of dP and D is nothing but roundings.)
    close_backward(got[2:], q, k, v, do, causal=causal, rows=slice(1 if causal else 0, None), axes=(-1,))


@pytest.mark.parametrize("shape", [(8, 12, 63, 64), (1, 2, 300, 64), (8, 16, 512, 64), (8, 12, 63, 128), (1, 2, 512, 128), (8, 16, 300, 128)],
                         ids=str)
def test_rows_of_dv_whose_keys_few_attend_to(dev, shape):
    """Every other key has logits 8 below the rest: its row of dV is made of probabilities of 2^-20 alone, which two halves still hold (further
    below, and dK: test_gpu_f32_lost_bits.py).  Held to itself: a logit of 8 is
    off by 2^-21 at most, its exponential by as much, and the probabilities' two halves end at 2^-39."""
    q, k, v, do = (synth.normal(77 + 10 ** 6 * i, shape) for i in range(4))
    q[..., 0] = 4
    k[..., 0] = 0
    k[..., ::2, 0] = -2.0 * np.sqrt(shape[3])
    got = run_fwd_bwd(dev, q, k, v, do)[4][:1, :2].astype(np.float64)
    want = oracle.attention_backward_f64(*(x[:1, :2].astype(np.float64) for x in (q, k, v, do)))[4]
    assert (np.linalg.norm(got - want, axis=-1) <= 2 * TOL * np.linalg.norm(want, axis=-1)).all()


@pytest.mark.parametrize("mode", ["plain", "causal", "causal+len"])
@pytest.mark.parametrize("shape", [(4, 12, 129, 128), (4, 12, 161, 128), (4, 12, 256, 128), (16, 16, 33, 128), (16, 16, 128, 128)], ids=str)
def test_tilings_of_head_size_128(dev, shape, mode):
    """128 queries per workgroup on few heads, 256 on many short ones, at the edges of their tiles."""
    B, H, N, D = shape
    q, k, v = (synth.normal(900 + 10 ** 6 * i, shape) for i in range(3))
    lens = ((np.arange(B) * 37 + 1) % (N + 1)).astype(np.int32) if "len" in mode else None
    got = run_flash(dev, q, k, v, F32, kv_len=lens, causal="causal" in mode)
    for b, h in ((0, 0), (B // 2, 3), (B - 1, H - 1)):
        want = oracle.sdpa_f64(q[b:b + 1, h:h + 1], k[b:b + 1, h:h + 1], v[b:b + 1, h:h + 1], causal="causal" in mode,
                               kv_len=None if lens is None else lens[b:b + 1])
        assert np.abs(got[b, h] - want[0, 0]).max() <= 3e-6 * np.abs(v[b, h]).max(), (b, h)
