"""The tilings of the fp32 kernels at the edges of their tiles, against the float64 oracle on sampled heads: many heads, so that
the launches take the tilings whose waves share their key (query) tiles and not the one for few, short heads."""
import numpy as np
import pytest

import oracle
from autorust_amd import synth
from autorust_amd.device import F32
from gpu_util import run_flash
from test_gpu_bwd import run_fwd_bwd

pytestmark = pytest.mark.gpu

# 256 heads: 128 queries per workgroup (last tile of one key, full tiles, waves without queries); 128 heads: 256 queries
SHAPES = [(16, 16, 65, 64), (16, 16, 97, 64), (16, 16, 128, 64), (16, 16, 33, 128), (16, 16, 65, 128), (16, 16, 128, 128),
          (8, 16, 257, 64), (8, 16, 289, 64), (8, 16, 384, 64), (8, 16, 257, 128), (8, 16, 320, 128)]


@pytest.mark.parametrize("mode", ["plain", "causal", "causal+len", "len"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_f32_forward_tilings(dev, shape, mode):
    B, H, N, D = shape
    # operands whose three bf16 parts all matter, over a few binary orders of magnitude
    q, k, v = (synth.normal(900 + i, (B, H, N, D)) for i in range(3))
    v *= np.exp2(np.arange(B, dtype=np.float32) - 8)[:, None, None, None]
    causal = "causal" in mode
    lens = ((np.arange(B) * 37 + 1) % (N + 1)).astype(np.int32) if "len" in mode else None
    got = run_flash(dev, q, k, v, F32, kv_len=lens, causal=causal)
    for b, h in ((0, 0), (B // 2, 3), (B - 1, H - 1)):
        want = oracle.sdpa_f64(q[b:b + 1, h:h + 1], k[b:b + 1, h:h + 1], v[b:b + 1, h:h + 1], causal=causal,
                               kv_len=None if lens is None else lens[b:b + 1]) if lens is None or lens[b] > 0 else np.zeros((1, 1, N, D))
        assert np.abs(got[b, h] - want[0, 0]).max() <= 3e-6 * max(np.abs(v[b, h]).max(), 1e-30), (b, h)


@pytest.mark.parametrize("mode", ["plain", "causal", "causal+len", "mask"])
@pytest.mark.parametrize("shape", [(16, 16, 16, 1, 64), (16, 8, 8, 33, 64), (8, 32, 16, 97, 64), (16, 8, 8, 129, 64), (16, 8, 8, 32, 128),
                                   (8, 16, 8, 65, 128), (8, 8, 8, 257, 128)], ids=str)
def test_f32_backward_tilings(dev, shape, mode):
    B, Hq, Hkv, N, D = shape
    q, do = (synth.normal(920 + i, (B, Hq, N, D)) for i in range(2))
    k, v = (synth.normal(930 + i, (B, Hkv, N, D)) for i in range(2))
    causal = "causal" in mode
    lens = (1 + (np.arange(B) * 37) % N).astype(np.int32) if "len" in mode else None
    mask = synth.normal(940, (N, N)) if mode == "mask" else None
    got = run_fwd_bwd(dev, q, k, v, do, mask=mask, kv_len=lens, causal=causal)
    g = Hq // Hkv
    for b, h in ((0, 0), (B - 1, Hkv - 1)):
        hs = slice(h * g, (h + 1) * g)
        want = oracle.attention_backward_f64(q[b:b + 1, hs], k[b:b + 1, h:h + 1], v[b:b + 1, h:h + 1], do[b:b + 1, hs], mask=mask,
                                             kv_len=None if lens is None else lens[b:b + 1], causal=causal)
        for name, x, w in zip(("o", "lse", "dq", "dk", "dv"), got, want):
            x = x[b:b + 1, hs] if name in ("o", "lse", "dq") else x[b:b + 1, h:h + 1]
            assert np.abs(x - w).max() <= 1e-5 * max(1.0, np.abs(w).max()), (name, b, h)


@pytest.mark.parametrize("shape", [(1, 4, 2, 1, 64), (1, 4, 2, 65, 64), (16, 8, 8, 33, 64), (16, 8, 8, 129, 64), (8, 32, 16, 97, 64),
                                   (16, 8, 8, 1, 128), (16, 8, 8, 65, 128), (8, 8, 8, 257, 128)], ids=str)
def test_f32_backward_tilings_causal_with_a_mask(dev, shape):
    """A causal launch with an additive mask that hides some keys: the mask of a tile is asked for ahead, in whole vectors except at
    the end of a row."""
    B, Hq, Hkv, N, D = shape
    q, do = (synth.normal(920 + 10 ** 6 * i, (B, Hq, N, D)) for i in range(2))
    k, v = (synth.normal(930 + 10 ** 6 * i, (B, Hkv, N, D)) for i in range(2))
    mask = synth.normal(940, (N, N))
    mask[:, N // 3] = -np.inf
    mask[N // 2, : N // 4] = -np.inf
    np.fill_diagonal(mask, 0.25)
    got = run_fwd_bwd(dev, q, k, v, do, mask=mask, causal=True)
    g = Hq // Hkv
    for b, h in ((0, 0), (B - 1, Hkv - 1)):
        hs = slice(h * g, (h + 1) * g)
        want = oracle.attention_backward_f64(q[b:b + 1, hs], k[b:b + 1, h:h + 1], v[b:b + 1, h:h + 1], do[b:b + 1, hs], mask=mask, causal=True)
        for name, x, w in zip(("o", "lse", "dq", "dk", "dv"), got, want):
            x = x[b:b + 1, hs] if name in ("o", "lse", "dq") else x[b:b + 1, h:h + 1]
            assert np.abs(x - w).max() <= 1e-5 * max(1.0, np.abs(w).max()), (name, b, h)
