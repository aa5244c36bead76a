"""Workloads that measure this framework: what they are, their inputs, one pass of each through the
public entry points, and the bytes and operations a pass cannot do without.

Five paths are covered, named by a case's "path":
  flash    Device.flash_fwd / flash_fwd_strided: fp32 exact and bf16 attention (causal, key lengths,
           additive mask, grouped-query heads, token-major layout)
  sage     Device.sage_quant (K smoothed and quantised) + Device.sage_fwd_qfused: int8 or FP8 attention
  train    Device.flash_fwd_lse + Device.flash_bwd: the fp32 training step, forward and backward
  tensor   Tensor.flash_attention_with on a Session: the tensor interface, exact or bf16 attention
  tensor_sage  Tensor.sage_attention_with: the tensor interface, quantised attention (f32 tensors with a
           scale per row and no smoothing, or bf16 tensors with block scales and smoothed K)
"""
import math

import numpy as np
import torch

from autorust_amd import host
from autorust_amd.device import BF16, F32, Device

_CACHE = {}


def _device():
    """One handle per process, as a program keeps it."""
    if "dev" not in _CACHE:
        _CACHE["dev"] = Device(0)
    return _CACHE["dev"]


def _host_device():
    if "host" not in _CACHE:
        _CACHE["host"] = host.HipDevice(0)
    return _CACHE["host"]


def _case(name, path, B, Hq, Hkv, N, D, dtype, causal=False, lens=False, mask=False, token_major=False, fp8=False, outliers=False):
    c = {"path": path, "B": B, "Hq": Hq, "Hkv": Hkv, "N": N, "D": D, "dtype": dtype, "causal": causal, "lens": lens, "mask": mask,
         "token_major": token_major, "fp8": fp8, "outliers": outliers}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # One image through a ViT-B/16 layer in exact mode: the smallest call, launch and latency.
        _case("vit_b1_f32", "flash", 1, 12, 12, 197, 64, "f32"),
        # A ViT-B/16 layer on a batch of images, the way a model calls it: tensors, a session, bf16.
        _case("vit_b8_bf16_tensor", "tensor", 8, 12, 12, 197, 64, "bf16"),
        # A small ViT on 448-pixel images in exact mode: the shape the reference quotes its kernels on.
        _case("vit_s_448px_f32", "flash", 8, 6, 6, 789, 64, "f32"),
        # The same layer quantised in the reference's own convention: f32 tensors, a scale per row.
        _case("vit_s_448px_sage_rows_tensor", "tensor_sage", 8, 6, 6, 789, 64, "f32"),
        # An encoder layer with a dense additive [N, N] bias (relative positions), bf16.
        _case("encoder_bias_bf16", "flash", 4, 16, 16, 1024, 64, "bf16", mask=True),
        # Prefill of a padded batch of prompts: causal with a key length per prompt.
        _case("decoder_prefill_bf16", "flash", 4, 32, 32, 2048, 128, "bf16", causal=True, lens=True),
        # Long prompts of a grouped-query model, straight from and to the projections' [B, N, H, D].
        _case("gqa_prefill_bf16", "flash", 2, 32, 8, 6150, 128, "bf16", causal=True, token_major=True),
        # The quantised forward on a long sequence: smoothed K, int8, no mask.
        _case("sage_s8192", "sage", 4, 32, 32, 8192, 128, "bf16"),
        # Causal quantised prefill with FP8 codes.
        _case("sage_fp8_causal_s4096", "sage", 2, 32, 32, 4096, 128, "bf16", causal=True, fp8=True),
        # Long-context causal quantised prefill on activations with outliers: the largest.
        _case("sage_causal_s32768", "sage", 1, 64, 64, 32768, 128, "bf16", causal=True, outliers=True),
        # Training step of a ViT-B/16 layer on a batch.
        _case("vit_b8_train_f32", "train", 8, 12, 12, 197, 64, "f32"),
        # Training step of a causal language-model layer.
        _case("lm_train_f32", "train", 2, 16, 16, 2048, 128, "f32", causal=True),
    ]


# flops of a drawn case, at most, by path and type: each takes less time than the largest listed case
_MOST = {"flash_f32": 0.4e12, "flash_bf16": 4e12, "sage": 8e12, "train": 0.4e12, "tensor_f32": 0.1e12, "tensor_bf16": 0.5e12,
         "tensor_sage": 0.5e12}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["flash", "flash", "flash", "sage", "sage", "train", "train", "tensor", "tensor_sage"])
    dtype = {"sage": "bf16", "train": "f32"}.get(path) or rng.choice(["f32", "bf16"])
    D = rng.choice([64, 128])
    causal = rng.random() < 0.5
    hi = {"flash": 16384, "sage": 32768, "train": 4096, "tensor": 2048, "tensor_sage": 2048}[path]
    N = _log_int(rng, 128 if path == "sage" else 16, hi)
    if rng.random() < 0.3:
        N = max(64, N // 64 * 64)
    B = _log_int(rng, 1, 16)
    Hq = rng.choice([4, 6, 8, 12, 16, 24, 32, 40])
    Hkv = Hq // 4 if Hq % 4 == 0 and rng.random() < 0.25 else Hq
    c = _case(None, path, B, Hq, Hkv, N, D, dtype, causal=causal)
    if path == "flash":
        c["lens"] = rng.random() < 0.3
        c["token_major"] = rng.random() < 0.3
        c["mask"] = N <= 4096 and rng.random() < 0.2
    if path == "sage":
        c["fp8"] = rng.random() < 0.3
        c["outliers"] = rng.random() < 0.3
    most = _MOST[path if path in ("sage", "train", "tensor_sage") else path + "_" + dtype]
    while work(c)["flops"] > most or c["B"] * c["Hq"] * c["N"] * c["D"] > (1 << 24 if path.startswith("tensor") else 1 << 28):
        if c["B"] > 1:
            c["B"] = (c["B"] + 1) // 2
        else:
            c["N"] = c["N"] * 3 // 4
    return c


def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


class _DeviceArray:
    """A tensor of the framework as device memory that torch can look at; keeps it alive."""

    def __init__(self, t, shape, typestr):
        self.t = t
        self.__cuda_array_interface__ = {"data": (host.host().arh_tensor_ptr(t.h), False), "shape": shape, "typestr": typestr,
                                         "strides": None, "version": 2}


def prepare(case, seed):
    c = dict(case)
    B, Hq, Hkv, N, D = c["B"], c["Hq"], c["Hkv"], c["N"], c["D"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    f32 = c["dtype"] == "f32"
    tm = c["token_major"]
    qshape, kshape = ((B, N, Hq, D), (B, N, Hkv, D)) if tm else ((B, Hq, N, D), (B, Hkv, N, D))
    q, k, v = _normal(gen, *qshape), _normal(gen, *kshape), _normal(gen, *kshape)
    if c["path"] in ("sage", "tensor_sage"):
        # keys carry a bias per channel; activations of long contexts have a few large entries
        k += _normal(gen, 1, Hkv, 1, D) * (5.0 if c["outliers"] else 3.0)
        if c["outliers"]:
            for x in (q, k):
                x *= torch.where(torch.rand(x.shape, generator=gen, device="cuda") < 0.01, 20.0, 1.0)
    if c["path"].startswith("tensor"):
        dev = _host_device()
        dt = host.FLOAT32 if f32 else host.BFLOAT16
        st = host.Settings.default()
        if c["path"] == "tensor_sage" and f32:
            st.sage_block_q = st.sage_block_k = 1
            st.sage_smooth_k = 0
        c.update(sess=host.Session(), settings=st, shape=qshape,
                 **{n: host.Tensor.from_slice(dev, t.cpu().numpy(), t.shape, dt) for n, t in (("q", q), ("k", k), ("v", v))})
        return c
    dtype = torch.float32 if f32 else torch.bfloat16
    c.update(dev=_device(), q=q.to(dtype), k=k.to(dtype), v=v.to(dtype), type=F32 if f32 else BF16)
    c["o"] = torch.empty(qshape, device="cuda", dtype=dtype)
    if c["lens"]:
        n = torch.randint((N + 1) // 2, N + 1, (B,), generator=gen, device="cuda")
        c["len"] = n.to(torch.int32)
    if c["mask"]:
        c["bias"] = _normal(gen, N, N)
    if tm:
        c["qs"], c["ks"] = (N * Hq * D, D, Hq * D), (N * Hkv * D, D, Hkv * D)
    if c["path"] == "sage":
        c["k8"] = torch.empty((B, Hkv, N, D), device="cuda", dtype=torch.uint8 if c["fp8"] else torch.int8)
        c["sk"] = torch.empty((B, Hkv, (N + 63) // 64), device="cuda", dtype=torch.float32)
        c["mean"] = torch.empty((B, Hkv, D), device="cuda", dtype=torch.float32)
        c["ws"] = torch.empty((max(4, c["dev"].sage_quant_workspace(B, Hkv, N, D)),), device="cuda", dtype=torch.uint8)
    if c["path"] == "train":
        c["dout"] = _normal(gen, *qshape)
        c["lse"] = torch.empty((B, Hq, N), device="cuda", dtype=torch.float32)
        c["delta"] = torch.empty((B, Hq, N), device="cuda", dtype=torch.float32)
        c["dq"], c["dk"], c["dv"] = (torch.empty_like(t) for t in (q, k, v))
    # the handle works on a stream of its own
    torch.cuda.synchronize()
    return c


def run(s):
    path = s["path"]
    if path.startswith("tensor"):
        fn = s["q"].sage_attention_with if path == "tensor_sage" else s["q"].flash_attention_with
        out = fn(s["k"], s["v"], None, 0.0, s["causal"], s["sess"], s["settings"])
        if s["dtype"] == "f32":
            return torch.as_tensor(_DeviceArray(out, s["shape"], "<f4"), device="cuda")
        return torch.as_tensor(_DeviceArray(out, s["shape"], "<i2"), device="cuda").view(torch.bfloat16)
    dev, B, Hq, Hkv, N, D, causal = s["dev"], s["B"], s["Hq"], s["Hkv"], s["N"], s["D"], s["causal"]
    q, k, v, o = s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["o"].data_ptr()
    if path == "flash":
        lens = s["len"].data_ptr() if s["lens"] else None
        bias = s["bias"].data_ptr() if s["mask"] else None
        if s["token_major"]:
            dev.flash_fwd_strided(q, k, v, o, s["qs"], s["ks"], s["qs"], B, Hq, Hkv, N, D, s["type"], mask=bias, kv_len=lens,
                                  causal=causal, wait=False)
        else:
            dev.flash_fwd(q, k, v, o, B, Hq, Hkv, N, D, s["type"], mask=bias, kv_len=lens, causal=causal, wait=False)
        return s["o"]
    if path == "sage":
        quant = dev.sage_quant_fp8 if s["fp8"] else dev.sage_quant
        quant(k, s["k8"].data_ptr(), s["sk"].data_ptr(), B, Hkv, N, D, 64, BF16, mean=s["mean"].data_ptr(),
              workspace=s["ws"].data_ptr(), smooth=True, wait=False)
        dev.sage_fwd_qfused(q, s["k8"].data_ptr(), s["sk"].data_ptr(), v, o, B, Hq, Hkv, N, D, 64, causal=causal, wait=False,
                            fp8=s["fp8"])
        return {"o": s["o"], "k8": s["k8"], "sk": s["sk"], "mean": s["mean"]}
    dev.flash_fwd_lse(q, k, v, o, s["lse"].data_ptr(), B, Hq, Hkv, N, D, F32, causal=causal, wait=False)
    dev.flash_bwd(q, k, v, o, s["lse"].data_ptr(), s["dout"].data_ptr(), s["dq"].data_ptr(), s["dk"].data_ptr(), s["dv"].data_ptr(),
                  s["delta"].data_ptr(), B, Hq, Hkv, N, D, causal=causal, wait=False)
    return {"o": s["o"], "lse": s["lse"], "dq": s["dq"], "dk": s["dk"], "dv": s["dv"]}


def work(case):
    B, Hq, Hkv, N, D = (case[x] for x in ("B", "Hq", "Hkv", "N", "D"))
    # visible (query, key) pairs of a head; key lengths are uniform in [N/2, N]
    if case["causal"]:
        pairs = N * (N + 1) / 2 if not case["lens"] else 11 / 24 * N * N
    else:
        pairs = N * N * (0.75 if case["lens"] else 1.0)
    es = 4 if case["dtype"] == "f32" else 2
    nbytes = (2 * Hq + 2 * Hkv) * B * N * D * es
    flops = 4.0 * B * Hq * D * pairs
    if case["mask"]:
        nbytes += 4 * N * N
    if case["path"] == "sage":
        # the codes and scales of K come out too
        nbytes += B * Hkv * (N * D + 4 * ((N + 63) // 64) + 4 * D)
    if case["path"] == "train":
        # forward 2 products, backward 5; in: q, k, v, dout; out: o, lse, dq, dk, dv
        nbytes = (4 * Hq + 4 * Hkv) * B * N * D * 4 + B * Hq * N * 4
        flops *= 3.5
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # quantised attention keeps its probabilities in bf16; whole values (codes) are the same
    if case["dtype"] == "bf16" or case["path"] in ("sage", "tensor_sage"):
        return {"rel": 1e-2, "differ": 0.0}
    return {"rel": 1e-5}
