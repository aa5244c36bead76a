"""Attention entries launched by name where arhip_launch takes another form than the entry's own: the results are those of the typed entry bit
for bit, which runs the same kernel."""
import numpy as np
import pytest

from autorust_amd import _lib, synth
from autorust_amd.device import BF16, F32
from gpu_util import Bufs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kernels(dev):
    return dev.module_load(open(_lib.KERNELS_PATH, "rb").read())


# entry, B, Hq, Hkv, N, D, causal, mask, key lengths: more workgroups than compute units, tilings of 256, 128 and 32 queries
F32_CASES = [
    ("ar_flash_f32", 8, 6, 6, 789, 64, False, False, None), ("ar_flash_f32", 8, 8, 4, 600, 64, True, True, None),
    ("ar_flash_f32_lens", 3, 24, 8, 650, 64, False, False, [650, 1, 0]), ("ar_flash_f32", 1, 8, 8, 1024, 128, False, False, None),
    ("ar_flash_f32_lens", 8, 16, 16, 300, 128, True, False, [300, 7, 0, 256, 257, 32, 33, 299]), ("ar_flash_f32_short", 4, 40, 40, 200, 64, False, False, None),
    ("ar_fl_fwd", 8, 6, 6, 789, 64, False, False, None), ("ar_fl_fwd", 1, 4, 2, 512, 128, False, True, None),
]


@pytest.mark.parametrize("case", F32_CASES, ids=str)
def test_f32(dev, kernels, case):
    name, B, Hq, Hkv, N, D, causal, has_mask, lens = case
    q, k, v = (synth.normal(s, (B, H, N, D)) for s, H in ((11, Hq), (12, Hkv), (13, Hkv)))
    rows = 32 if name.endswith("_short") else 128
    with Bufs(dev) as bufs:
        dq, dk, dv = (bufs.put(x) for x in (q, k, v))
        o, o2, lse, lse2 = bufs.new(q.nbytes), bufs.new(q.nbytes), bufs.new(B * Hq * N * 4), bufs.new(B * Hq * N * 4)
        dm = bufs.put(synth.normal(14, (N, N))) if has_mask else None
        dl = bufs.put(np.array(lens, np.int32)) if lens else None
        args = [dq, dk, dv, o] + ([lse] if name.startswith("ar_fl_") else []) + [dm or o] + ([dl] if lens else [])
        dev.launch(kernels, name, ((N + rows - 1) // rows, B * Hq, 1), (256, 1, 1), args, [N, D, int(causal), int(has_mask), Hq, Hkv])
        dev.flash_fwd_lse(dq, dk, dv, o2, lse2, B, Hq, Hkv, N, D, F32, mask=dm, kv_len=dl, causal=causal)
        assert o.copyout(np.float32, q.shape).tobytes() == o2.copyout(np.float32, q.shape).tobytes()
        if name.startswith("ar_fl_"):
            assert lse.copyout(np.float32, q.shape[:3]).tobytes() == lse2.copyout(np.float32, q.shape[:3]).tobytes()


@pytest.mark.parametrize("case", [c for c in F32_CASES if c[0] == "ar_flash_f32" and not c[7]], ids=str)
def test_a_module_of_the_callers(dev, case):
    """A kernel of one of these names in another module is the one that runs, also where the library's entry would take another form."""
    probes = dev.module_load(open(_lib.PROBES_PATH, "rb").read())
    name, B, Hq, Hkv, N, D = case[:6]
    with Bufs(dev) as bufs:
        o = bufs.new(B * Hq * N * D * 4)
        dev.launch(probes, name, ((N + 127) // 128, B * Hq, 1), (256, 1, 1), [o, o, o, o, o], [N, D, 0, 0, Hq, Hkv])
        got = o.copyout(np.float32, (B * Hq, N, D))
        assert (got == np.arange(N, dtype=np.float32)[:, None]).all()


# two groups of waves: 2 + 2 on 64 queries, 4 + 4 on 128
PIPE_CASES = [(1, 8, 2, 1000, 64, False, None), (2, 4, 4, 513, 128, True, [513, 70]), (1, 16, 16, 2048, 64, False, None), (1, 16, 16, 2047, 128, True, None)]


@pytest.mark.parametrize("kind", ["bf16", "int8", "fp8"])
@pytest.mark.parametrize("case", PIPE_CASES, ids=str)
def test_two_groups(dev, kernels, case, kind):
    B, Hq, Hkv, N, D, causal, lens = case
    q, k, v = (synth.normal(s, (B, H, N, D)) for s, H in ((21, Hq), (22, Hkv), (23, Hkv)))
    sfx = "_lens" if lens else ""
    with Bufs(dev) as bufs:
        dq, dk, dv = (bufs.put(synth.to_bf16_bits(x)) for x in (q, k, v))
        dl = bufs.put(np.array(lens, np.int32)) if lens else None
        o, o2 = bufs.new(q.nbytes), bufs.new(q.nbytes)
        grid, vals = ((N + 127) // 128, B * Hq, 1), [N, D, int(causal), 0, Hq, Hkv]
        if kind == "bf16":
            dev.launch(kernels, "ar_flash_bf16_mid" + sfx, grid, (256, 1, 1), [dq, dk, dv, o, o] + ([dl] if lens else []), vals)
            dev.flash_fwd(dq, dk, dv, o2, B, Hq, Hkv, N, D, BF16, kv_len=dl, causal=causal)
        else:
            fp8 = kind == "fp8"
            k8, sk, mean = bufs.new(k.size), bufs.new(B * Hkv * ((N + 63) // 64) * 4), bufs.new(B * Hkv * D * 4)
            ws = bufs.new(max(4, dev.sage_quant_workspace(B, Hkv, N, D)))
            (dev.sage_quant_fp8 if fp8 else dev.sage_quant)(dk, k8, sk, B, Hkv, N, D, 64, BF16, mean=mean, workspace=ws, smooth=True)
            sq, sq2 = bufs.new(B * Hq * ((N + 127) // 128) * 4), bufs.new(B * Hq * ((N + 127) // 128) * 4)
            name = ("ar_flash_sage_fp8_qf_mid" if fp8 else "ar_flash_sage_qf_mid") + sfx
            dev.launch(kernels, name, grid, (256, 1, 1), [dq, k8, dv, o, o] + ([dl] if lens else []) + [sq, sk], vals + [128, 64, 1])
            dev.sage_fwd_qfused(dq, k8, sk, dv, o2, B, Hq, Hkv, N, D, 64, out_dtype=F32, sq_out=sq2, kv_len=dl, causal=causal, fp8=fp8)
            assert sq.copyout(np.float32, (sq.nbytes // 4,)).tobytes() == sq2.copyout(np.float32, (sq2.nbytes // 4,)).tobytes()
        assert o.copyout(np.uint8, (q.nbytes,)).tobytes() == o2.copyout(np.uint8, (q.nbytes,)).tobytes()
