"""Device buffers that are handed out again, ids and results that pass through the library's pinned memory (csrc/runtime.hip)."""
import numpy as np
import pytest

from webgpt_amd import _lib, blocks

import ctypes as C

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(7)


@pytest.mark.parametrize("n", [4, 1020, 1024, 262140, 262144, 262148, 400000])
def test_downloads_of_any_length_and_offset(device, n):
    """On both sides of the megabyte that goes through pinned memory, and parts that are no multiple of 16 bytes."""
    a = RNG.standard_normal(n).astype(np.float32)
    b = blocks.init_tensor(a, [n])
    assert np.array_equal(b.download(), a)
    for offset, count in ((4, 1), (16, n - 4), (8, n - 3), (0, n - 1)):
        if count > 0:
            assert np.array_equal(b.download(count=count, offset=offset), a[offset // 4:offset // 4 + count])
    b.destroy()


def test_buffers_freed_under_launches_that_read_them(device):
    """Buffers that the host has not written to (which the library keeps) given back and handed out again at once, and written by a later
    launch, while the launch that reads them waits its turn on the stream: nothing in between uploads, downloads or waits."""
    n, rounds = 1 << 20, 100
    a, b = (RNG.standard_normal(n).astype(np.float32) for _ in range(2))
    xa, xb = blocks.init_tensor(a, [n]), blocks.init_tensor(b, [n])
    slow = [blocks.Buffer([16 * n]) for _ in range(2)]

    def add(x, y, out, count=n):
        _lib.call("wgpt_residual", 1, count, x.handle, y.handle, out.handle)

    outs = []
    for i in range(rounds):
        if i % 10 == 0:  # (the launches of ten rounds take the device longer than the host)
            for _ in range(8):
                add(slow[0], slow[0], slow[1], 16 * n)
        first, out = blocks.Buffer([n]), blocks.Buffer([n])
        add(xa, xb if i % 2 else xa, first)
        add(first, xb, out)
        first.destroy()
        again = blocks.Buffer([n])  # (a block of this size is there: the one that the launch above reads)
        add(xb, xb, again)
        again.destroy()
        outs.append(out)
        if len(outs) > 12:  # (so are results that nobody has asked for)
            outs.pop(0).destroy()
    for i, out in list(zip(range(rounds), [None] * (rounds - len(outs)) + outs)):
        if out:
            assert np.array_equal(out.download(), (a + (b if i % 2 else a)) + b), i
            out.destroy()
    for x in [xa, xb] + slow:
        x.destroy()


def test_ids_of_many_embeddings_under_way(device):
    """More ids than the pinned ring holds, and a call with more than all of it, without a wait in between."""
    V, d = 97, 8
    wte, wpe = RNG.standard_normal((V, d)).astype(np.float32), RNG.standard_normal((20000, d)).astype(np.float32)
    bt, bp = blocks.init_tensor(wte, [V, d]), blocks.init_tensor(wpe, [20000, d])
    calls = []
    for T in [3000] * 12 + [16384, 20000, 1]:
        ids = RNG.integers(0, V, T).astype(np.int32)
        out = blocks.Buffer([T, d])
        passed = ids.copy()
        _lib.call("wgpt_embed", passed.ctypes.data_as(C.POINTER(C.c_int32)), T, d, V, bt.handle, bp.handle, out.handle)
        passed[:] = 0  # the caller's memory is the caller's again
        calls.append((ids, out))
    for ids, out in calls:
        assert np.array_equal(out.download().reshape(-1, d), wte[ids] + wpe[:len(ids)])
        out.destroy()
    bt.destroy()
    bp.destroy()
