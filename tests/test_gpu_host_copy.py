"""Copies between host arrays and the device (host_copy.cpp): every size class and its edges, byte for byte, against
the array itself; inputs of a session that are queued behind each other."""
import threading

import numpy as np
import pytest

from meganeura_amd import capi
from meganeura_amd.graph import Graph, build_inference_session

pytestmark = pytest.mark.gpu

CHUNK, SLOT, SMALL = 1 << 20, 2 << 20, 4 << 20  # host_copy.cpp: kChunk, kSlot and kSmallIn, kSmall; kLargeIn is 8 slots
SIZES = [1, 3, 4, 2304, (512 << 10) - 1, 512 << 10, (512 << 10) + 1, CHUNK + 1, SLOT, SLOT + 1, SMALL - 1, SMALL, SMALL + 1, 5 * SLOT, 8 * SLOT - 1, 8 * SLOT, 8 * SLOT + 7, 33 * SLOT - 5]


def pattern(nbytes, seed):
    return np.random.default_rng(seed).integers(0, 256, nbytes, dtype=np.uint8)


@pytest.mark.parametrize("nbytes", SIZES)
def test_round_trip(nbytes):
    with capi.Context(0) as ctx:
        for offset, seed in ((0, 1), (13, 2)):
            b = ctx.buffer(nbytes + 64)
            want = pattern(nbytes, seed)
            b.upload(want, offset)
            assert np.array_equal(b.download(np.uint8, nbytes, offset), want)
            assert not b.download(np.uint8, 64 - offset, nbytes + offset).any(), "nothing written past the end"
            b.free()


def test_ring_wraps():
    """More uploads than the pinned ring holds, and nothing overwritten before it has travelled."""
    with capi.Context(0) as ctx:
        bufs = [(ctx.buffer(3 << 20), pattern(3 << 20, s)) for s in range(8)]
        for b, want in bufs:
            b.upload(want)
        for b, want in bufs:
            assert np.array_equal(b.download(np.uint8, want.size), want)


def test_queued_inputs():
    """set_input returns before the bytes have arrived: the caller's array may change at once, and inputs that
    together exceed the ring (16 MiB) still all arrive before the step."""
    m, k = 1536, 1024  # 6 MiB each
    g = Graph()
    x, y = g.input("x", [m, k]), g.input("y", [m, k])
    g.set_outputs([g.add(x, y)])
    s = build_inference_session(g)
    scratch = np.empty((m, k), np.float32)
    for step in range(5):
        scratch[:] = step
        s.set_input("x", scratch)
        scratch[:] = 10 * step
        s.set_input("y", scratch)
        scratch[:] = -1
        if step % 2:
            s.set_input("x", np.full((m, k), 100.0, np.float32))
        s.step()
        s.wait()
        want = (100.0 if step % 2 else step) + 10.0 * step
        assert (s.read_output(m * k) == want).all()
    s.close()


def test_contexts_on_threads():
    """Each thread with a context of its own: large and small copies side by side."""
    bad = []

    def work(seed):
        with capi.Context(0) as ctx:
            for i, nbytes in enumerate((9 * SLOT, 1000, SMALL, 6 * SLOT + 1)):
                want = pattern(nbytes, 10 * seed + i)
                b = ctx.buffer(nbytes)
                b.upload(want)
                if not np.array_equal(b.download(np.uint8, nbytes), want):
                    bad.append((seed, nbytes))
                b.free()

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad
