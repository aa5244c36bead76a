"""What the C++ host layer submits and waits for (csrc/host/): a launch is submitted without waiting only while everything that can see its
buffers goes to the same stream.  CPU tests: the host layer on a stand-in for libarhip that logs launches and waits.  GPU tests:
results read through the address on another stream, and buffers shared between two handles."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from autorust_amd import host, synth
from autorust_amd.host import BFLOAT16, FLOAT32, Session, Settings, Tensor

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "..", "autorust_amd", "csrc", "host")


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("host_stub")
    lib = str(tmp / "libstub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-o", lib, os.path.join(HERE, "host_stub.cpp"),
                    os.path.join(SRC, "autorust_host.cpp"), os.path.join(SRC, "host_capi.cpp"), "-ldl"], check=True)
    kernels = tmp / "kernels.bin"
    kernels.write_bytes(b"none")
    os.environ["AUTORUST_HIP_KERNELS"] = str(kernels)
    h = ctypes.CDLL(lib)
    for f in ("arh_device_open", "arh_tensor_from_slice", "arh_session_new", "arh_attention", "arh_tensor_ptr"):
        getattr(h, f).restype = ctypes.c_void_p
    h.stub_log.restype = ctypes.c_char_p
    yield h
    del os.environ["AUTORUST_HIP_KERNELS"]


class _Stub:
    """The few calls of the host layer's C view that the tests make, by raw handles."""

    def __init__(self, h):
        self.h, self.sess = h, ctypes.c_void_p(h.arh_session_new())

    def device(self):
        return ctypes.c_void_p(self.h.arh_device_open(0))

    def tensor(self, dev, dtype=FLOAT32, shape=(1, 2, 64, 64)):
        x = np.zeros(shape, np.float32)
        dims = (ctypes.c_int64 * len(shape))(*shape)
        return ctypes.c_void_p(self.h.arh_tensor_from_slice(dev, x.ctypes.data_as(ctypes.c_void_p), dims, len(shape), dtype))

    def attention(self, q, k, v, api=2, mask=None, causal=False):
        """The new tensor and the log of the call."""
        self.h.stub_clear()
        out = self.h.arh_attention(q, k, v, mask, ctypes.c_double(0.0), int(causal), api, self.sess, None, None)
        assert out
        return ctypes.c_void_p(out), self.h.stub_log().decode().split("\n")[:-1]


def test_calls_on_one_handle_do_not_wait(stub):
    s = _Stub(stub)
    d = s.device()
    q, k, v = (s.tensor(d) for _ in range(3))
    _, log = s.attention(q, k, v)
    assert log and all(line.startswith("launch ") for line in log)


def test_an_address_is_handed_out_after_the_work_on_it(stub):
    s = _Stub(stub)
    d = s.device()
    q, k, v = (s.tensor(d) for _ in range(3))
    out, log = s.attention(q, k, v)
    me = log[0].split()[1]
    stub.stub_clear()
    assert stub.arh_tensor_ptr(out)
    assert stub.stub_log().decode() == "sync %s\n" % me


@pytest.mark.parametrize("which", ["read", "written"])
def test_launches_on_a_buffer_whose_address_is_out_are_waited_for(stub, which):
    s = _Stub(stub)
    d = s.device()
    q, k, v = (s.tensor(d) for _ in range(3))
    if which == "read":
        stub.arh_tensor_ptr(k)
        _, log = s.attention(q, k, v)
    else:
        stub.arh_session_begin_capture(s.sess)
        out, _ = s.attention(q, k, v)
        assert stub.arh_session_end_capture(s.sess) == 1
        stub.arh_tensor_ptr(out)
        stub.stub_clear()
        stub.arh_session_replay(s.sess)
        log = stub.stub_log().decode().split("\n")[:-1]
    assert len(log) == 2 and log[0].startswith("launch ") and log[1] == "sync " + log[0].split()[1]


@pytest.mark.parametrize("api,dtype", [(2, FLOAT32), (3, FLOAT32), (3, BFLOAT16)])
@pytest.mark.parametrize("foreign", ["q", "k", "v"])
def test_buffers_of_another_handle_are_waited_for_on_both_sides(stub, api, dtype, foreign):
    """Every launch that touches a buffer of a handle other than its own runs between a wait for that handle's stream and a
    wait for its own."""
    s = _Stub(stub)
    a, b = s.device(), s.device()
    q, k, v = (s.tensor(b if n == foreign else a, dtype) for n in ("q", "k", "v"))
    _, log = s.attention(q, k, v, api)
    handles = {line.split()[1] for line in log}
    assert len(handles) == 2, log
    mixed = [i for i, line in enumerate(log) if line.endswith(" foreign")]
    assert mixed, log
    for i in mixed:
        me = log[i].split()[1]
        (other,) = handles - {me}
        assert log[i - 1] == "sync " + other and log[i + 1] == "sync " + me, log


# B, H, N (on 256 compute units), and whether the 32-query entry serves them: plain, causal, masked, causal and masked
@pytest.mark.parametrize("shape,short", [((4, 8, 512), (1, 1, 1, 1)), ((2, 12, 1024), (0, 1, 1, 1)), ((8, 8, 512), (0, 1, 1, 1)),
                                         ((8, 6, 789), (0, 0, 1, 1)), ((8, 16, 512), (0, 0, 0, 1)), ((8, 16, 640), (0, 0, 0, 0))])
def test_entry_of_the_fp32_forward(stub, shape, short):
    s = _Stub(stub)
    d = s.device()
    x = s.tensor(d, shape=shape + (64,))
    m = s.tensor(d, shape=(shape[2], shape[2]))
    for want, mask, causal in zip(short, (None, None, m, m), (False, True, False, True)):
        out, log = s.attention(x, x, x, mask=mask, causal=causal)
        assert [line.split()[2] for line in log] == ["ar_flash_f32_short" if want else "ar_flash_f32"], (causal, mask)
        stub.arh_tensor_free(out)
    for t in (x, m):
        stub.arh_tensor_free(t)


@pytest.mark.parametrize("shape,causal,short", [((1, 12, 1024), False, True), ((4, 8, 512), False, False), ((4, 8, 512), True, True),
                                                ((1, 8, 2048), True, True), ((2, 12, 700), True, False)])
def test_entries_of_the_fp32_backward(stub, shape, causal, short):
    s = _Stub(stub)
    d = s.device()
    x, lse = s.tensor(d, shape=shape + (64,)), s.tensor(d, shape=(shape[0] * shape[1], shape[2]))
    grads = [ctypes.c_void_p() for _ in range(3)]
    stub.stub_clear()
    assert stub.arh_fused_attention_backward(x, x, x, x, lse, x, None, int(causal), s.sess, *(ctypes.byref(g) for g in grads)) == 1
    names = [line.split()[2] for line in stub.stub_log().decode().split("\n")[:-1]]
    assert names == ["ar_fl_prep"] + [n + "_short" * short for n in ("ar_fl_bwd_dq", "ar_fl_bwd_dkv")]
    for t in [x, lse] + grads:
        stub.arh_tensor_free(t)


def _arrays(b=2, h=4, n=300, d=64):
    return [synth.normal(s, (b, h, n, d)) for s in (1, 2, 3)]


@pytest.mark.gpu
def test_an_address_is_good_on_any_stream(dev):
    """A tensor's memory read and cleared through its address on the stream of another handle, after the call that made it and
    after every replay into it."""
    from autorust_amd._lib import check
    hdev, sess = host.HipDevice(0), Session()
    q, k, v = (Tensor.from_slice(hdev, x, x.shape) for x in _arrays())
    want = q.flash_attention_with(k, v, None, 0.0, False, sess).to_list()
    sess.begin_capture()
    out = q.flash_attention_with(k, v, None, 0.0, False, sess)
    sess.end_capture()
    address = host.host().arh_tensor_ptr(out.h)
    got = np.empty_like(want)

    def read():
        check(dev.lib.arhip_copyout(dev.handle, got.ctypes.data, address, got.nbytes))
        return got

    assert np.array_equal(read(), want)
    for _ in range(3):
        check(dev.lib.arhip_fill_zero(dev.handle, address, got.nbytes))
        dev.sync()
        assert not read().any()
        sess.replay()
        assert np.array_equal(read(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("api", ["flash_attention_with", "sage_attention_with"])
def test_tensors_of_two_handles(api):
    """K made by a call on one handle and used by the next call on another at once, with the first handle's buffers reused
    behind it: the results of one handle."""
    a, b, sess, st = host.HipDevice(0), host.HipDevice(0), Session(), Settings.default()
    q, k, v = _arrays(n=1000)

    def chain(first, second):
        tq, tk, tv = (Tensor.from_slice(first, x, x.shape) for x in (q, k, v))
        q2 = Tensor.from_slice(second, q, q.shape)
        k2 = getattr(tq, api)(tk, tv, None, 0.0, False, sess, st)
        out = getattr(q2, api)(k2, tv, None, 0.0, False, sess, st)
        del k2
        getattr(tq, api)(tv, tk, None, 0.0, False, sess, st)     # takes the block that k2 left
        return out.to_list()

    want = chain(a, a)
    for _ in range(3):
        assert np.array_equal(chain(a, b), want)


@pytest.mark.gpu
def test_sync_and_stream_of_a_handle():
    dev = host.HipDevice(0)
    assert dev.stream
    dev.sync()
