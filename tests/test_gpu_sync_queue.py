"""arhip_sync behind a queue whose last piece alone writes what is looked at, by another handle, on a stream that nothing orders: queues that end while
the host looks for its number and queues that outlast the look, several threads on a handle, and copies that a caller put on the stream by
itself.  All but the threads also look before they wait, and have to have found the old value then: the queue is long enough to tell."""
import ctypes
import threading

import numpy as np
import pytest

from autorust_amd import synth
from autorust_amd._lib import check
from autorust_amd.device import F32, Device
from gpu_util import Bufs

pytestmark = pytest.mark.gpu
WORDS = 64
LOOKERS = 5  # handles that look, in turn: streams share the four hardware queues, and one on the queue of the work always comes behind it


@pytest.fixture
def lookers():
    got = [Device(0) for _ in range(LOOKERS)]
    yield got
    for d in got:
        d.close()


class _Queue:
    """`passes` attentions over H heads of N tokens, then a copy of row i of a table to the place that is looked at."""

    def __init__(self, dev, bufs, H, N, passes):
        self.dev, self.dims, self.passes = dev, (1, H, H, N, 64), passes
        x = synth.normal(61, (1, H, N, 64))
        self.x, self.o = bufs.put(x), bufs.new(x.nbytes)
        self.table = bufs.put(np.repeat(np.arange(1, 257, dtype=np.float32)[:, None], WORDS, axis=1))
        self.out = bufs.new(WORDS * 4)

    def submit(self, i):
        for _ in range(self.passes):
            self.dev.flash_fwd(self.x, self.x, self.x, self.o, *self.dims, F32, wait=False)
        check(self.dev.lib.arhip_copy_d2d(self.dev.handle, self.out.ptr, self.table.ptr + i * WORDS * 4, WORDS * 4))

    def seen_by(self, other):
        got = np.empty(WORDS, np.float32)
        check(other.lib.arhip_copyout(other.handle, got.ctypes.data, self.out.ptr, got.nbytes))
        return got

    def seconds(self):
        for _ in range(2):
            self.dev.timer_start()
            self.submit(0)
            secs = self.dev.timer_stop()
        return secs


# (the look takes 300 us)
@pytest.mark.parametrize("H,N,passes,least,most", [(8, 4096, 1, 5e-5, 2.9e-4), (24, 8192, 3, 1.5e-3, 1.0)], ids=["within the look", "beyond the look"])
def test_the_last_of_a_queue_is_there(dev, lookers, H, N, passes, least, most):
    with Bufs(dev) as bufs:
        queue = _Queue(dev, bufs, H, N, passes)
        assert least < queue.seconds() < most
        early = 0
        for i in range(1, 41):
            other = lookers[i % LOOKERS]
            queue.submit(i)
            if i % 2:
                early += (queue.seen_by(other) == np.float32(i)).all()
            dev.sync()
            assert (queue.seen_by(other) == np.float32(i + 1)).all(), i
        assert early >= 1


def test_threads_with_queues_on_a_handle(dev):
    others, wrong = [Device(0) for _ in range(3)], []
    with Bufs(dev) as bufs:
        queues = [_Queue(dev, bufs, 8, 2048, 1) for _ in others]

        def go(n):
            for i in range(1, 60):
                queues[n].submit(i)
                dev.sync()
                if not (queues[n].seen_by(others[n]) == np.float32(i + 1)).all():
                    wrong.append((n, i))

        threads = [threading.Thread(target=go, args=(n,)) for n in range(len(others))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    for d in others:
        d.close()
    assert not wrong


def test_copies_that_a_caller_put_on_the_stream(lookers):
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipMemcpyAsync.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int, ctypes.c_void_p]
    dev = Device(0)
    try:
        with Bufs(dev) as bufs:
            n = 256 << 20
            a, b, queue = bufs.new(n), bufs.new(n), _Queue(dev, bufs, 8, 64, 0)
            queue.submit(0)
            dev.sync()
            stream, early = dev.lib.arhip_stream(dev.handle), 0
            for i in range(1, 21):
                other = lookers[i % LOOKERS]
                for _ in range(20):
                    assert hip.hipMemcpyAsync(b.ptr, a.ptr, n, 3, stream) == 0  # device to device
                assert hip.hipMemcpyAsync(queue.out.ptr, queue.table.ptr + i * WORDS * 4, WORDS * 4, 3, stream) == 0
                if i % 2:
                    early += (queue.seen_by(other) == np.float32(i)).all()
                dev.sync()
                assert (queue.seen_by(other) == np.float32(i + 1)).all(), i
            assert early >= 1
    finally:
        dev.close()
