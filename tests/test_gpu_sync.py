"""arhip_sync: what was issued before it is done, whoever looks next: short work, work longer than the look for its number, several threads on
a handle, and a handle whose stream others use."""
import ctypes
import threading

import numpy as np
import pytest

from autorust_amd import synth
from autorust_amd._lib import check
from autorust_amd.device import F32, Device
from gpu_util import Bufs

pytestmark = pytest.mark.gpu


class _Work:
    """One query-independent attention: with a single key O is V, so every pass has another known result; rounds repeat it, to take longer."""

    def __init__(self, dev, bufs, B, H, D=64):
        self.dev, self.shape = dev, (B, H, 1, D)
        x = synth.normal(41, self.shape)
        self.q, self.k, self.v, self.o = bufs.put(x), bufs.put(x), bufs.put(x), bufs.new(x.nbytes)

    def run(self, value, rounds=1):
        self.v.copyin(np.full(self.shape, value, np.float32))
        B, H, N, D = self.shape
        for _ in range(rounds):
            self.dev.flash_fwd(self.q, self.k, self.v, self.o, B, H, H, N, D, F32, wait=False)


def _seen_by(other, work):
    out = np.empty(work.shape, np.float32)
    check(other.lib.arhip_copyout(other.handle, out.ctypes.data, work.o.ptr, out.nbytes))
    return out


@pytest.mark.parametrize("rounds", [1, 400])
def test_results_are_there_for_another_stream(dev, rounds):
    other = Device(0)
    try:
        with Bufs(dev) as bufs:
            w = _Work(dev, bufs, 64, 64)
            for i in range(40 if rounds == 1 else 5):
                w.run(float(i + 1), rounds)
                dev.sync()
                dev.sync()  # nothing more to wait for
                assert (_seen_by(other, w) == np.float32(i + 1)).all(), i
    finally:
        other.close()


def test_threads_on_a_handle(dev):
    other, wrong = [Device(0) for _ in range(3)], []
    with Bufs(dev) as bufs:
        works = [_Work(dev, bufs, 16, 16) for _ in other]

        def go(n):
            for i in range(60):
                works[n].run(float(100 * n + i + 1))
                dev.sync()
                if not (_seen_by(other[n], works[n]) == np.float32(100 * n + i + 1)).all():
                    wrong.append((n, i))

        threads = [threading.Thread(target=go, args=(n,)) for n in range(len(other))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    for d in other:
        d.close()
    assert not wrong


def test_work_of_others_on_the_stream():
    """Work that a caller puts on the handle's stream by itself is waited for too."""
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipMemcpyAsync.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int, ctypes.c_void_p]
    dev, other = Device(0), Device(0)
    try:
        with Bufs(dev) as bufs:
            n = 64 << 20
            a, b = bufs.put(np.full(n // 4, 7.0, np.float32)), bufs.new(n)
            dev.sync()
            stream = dev.lib.arhip_stream(dev.handle)
            assert hip.hipMemcpyAsync(b.ptr, a.ptr, n, 3, stream) == 0  # device to device
            dev.sync()
            out = np.empty(n // 4, np.float32)
            check(other.lib.arhip_copyout(other.handle, out.ctypes.data, b.ptr, n))
            assert (out == 7.0).all()
    finally:
        dev.close()
        other.close()
