"""The mean that smoothing subtracts, from 1 to 40 partial sums of 64 tokens: summed in LDS, at the head of the quantising workgroups or by a launch of
its own, in the same order and to the same bits."""
import numpy as np
import pytest

from autorust_amd import synth
from autorust_amd.device import BF16, F32
from gpu_util import Bufs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("chunks", [1, 2, 4, 5, 7, 8, 9, 15, 16, 17, 31, 32, 33, 40])
def test_mean(dev, chunks, D, dtype):
    B, H, N = 1, 4, 64 * chunks - 13
    x = synth.normal(975, (B, H, N, D)) + np.float32(2.0)
    if dtype == BF16:
        x = synth.from_bf16_bits(synth.to_bf16_bits(x))
    want = np.zeros((B, H, D), np.float32)
    for c in range(chunks):
        part = np.zeros((B, H, D), np.float32)
        for r in range(64 * c, min(64 * c + 64, N)):
            part = part + x[:, :, r]
        want = want + part
    want = want / np.float32(N)
    for block in (64, 128, 1):
        with Bufs(dev) as bufs:
            x8, sc, mean = bufs.new(x.size), bufs.new(B * H * ((N + block - 1) // block) * 4), bufs.new(B * H * D * 4)
            ws = bufs.new(dev.sage_quant_workspace(B, H, N, D))
            dev.sage_quant(bufs.put(synth.to_bf16_bits(x) if dtype == BF16 else x), x8, sc, B, H, N, D, block, dtype, mean=mean, workspace=ws, smooth=True)
            assert np.array_equal(mean.copyout(np.float32, want.shape), want), block
