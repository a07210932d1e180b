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
    """Freed at once, handed out again and written while the launches that read them wait their turn on the stream."""
    n = 1 << 20
    ins, outs = [], []
    for i in range(40):
        a = RNG.standard_normal(n).astype(np.float32)
        x, y = blocks.init_tensor(a, [n]), blocks.Buffer([n])
        _lib.call("wgpt_residual", 1, n, x.handle, x.handle, y.handle)
        x.destroy()
        ins.append(a)
        outs.append(y)
        if i >= 20:
            outs[i - 20].destroy()
    for a, y in list(zip(ins, outs))[20:]:
        assert np.array_equal(y.download(), a + a)
        y.destroy()


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
