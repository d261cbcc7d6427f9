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
    """Inputs go through the pinned ring without being waited for: more of them than it holds (16 MiB) in front of one step, pieces of
    odd lengths, the caller's array changing as soon as set_input returns, and of two writes to an input the later one."""
    m, k, count = 509, 1023, 12  # 2.08 MB each, just below the largest that takes this way
    assert (2 << 20) - (16 << 10) < m * k * 4 <= SLOT
    g = Graph()
    total = g.input("x0", [m, k])
    for i in range(1, count):
        total = g.add(total, g.input(f"x{i}", [m, k]))
    g.set_outputs([total])
    s = build_inference_session(g)
    scratch, ramp = np.empty((m, k), np.float32), np.arange(m * k, dtype=np.float32).reshape(m, k)
    for step in range(3):
        for round_ in range(2):
            for i in np.random.default_rng(10 * step + round_).permutation(count):
                scratch[:] = ramp * np.float32(i) + np.float32(step + 100 * round_)  # (whole numbers below 2^24: exact)
                s.set_input(f"x{i}", scratch)
                scratch[:] = -1
        s.step()
        s.wait()
        want = ramp.astype(np.float64) * sum(range(count)) + count * (step + 100)
        assert np.abs(s.read_output(m * k).reshape(m, k) - want).max() <= 2.0**-24 * count * want.max()
    s.close()


@pytest.mark.parametrize("m", [256, 1536])  # 1 MiB each, through the ring; 6 MiB, as the runtime copies
def test_queued_inputs(m):
    """set_input returns before the step that reads the bytes: the caller's array may change at once."""
    k = 1024
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
