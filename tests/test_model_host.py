"""Host code of the model entry points on tests/host_hip.cc, which stands in for the HIP runtime: kernels do not run, so only
error paths and the order of calls are looked at. A process of its own per test: the stand-in has to be loaded first."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes as C, sys
hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
launches, fail_at, unwaited = (C.c_int.in_dll(hip, "host_hip_" + n) for n in ("launches", "fail_at", "unwaited"))
allocs, alloc_fail_at = (C.c_int.in_dll(hip, "host_hip_" + n) for n in ("allocs", "alloc_fail_at"))
import numpy as np
from webgpt_amd import WgptError, _lib, synth
from helpers import make_model, small_cfg
_lib.init(0)
cfg = small_cfg(dtype=sys.argv[2])
tensors = make_model(cfg, 1)

def refused(name, *args):
    try:
        _lib.call(name, *args)
    except WgptError as e:
        return str(e) or "refused"
    return None

def model():
    m = C.c_uint64(0)
    _lib.call("wgpt_model_create", C.byref(_lib.Params(**synth.model_params(cfg), weight_dtype=int(sys.argv[2] == "int8"))), C.byref(m))
    for n, t in tensors.items():
        _lib.call("wgpt_model_set_tensor", m, n.encode(), np.ascontiguousarray(t).ctypes.data, t.nbytes)
    return m
"""


@pytest.fixture(scope="module")
def host_hip(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host_hip") / "host_hip.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-Wno-deprecated-declarations",
                    os.path.join(HERE, "host_hip.cc"), "-o", out], check=True)
    return out


def run(host_hip, dtype, body):
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([os.path.dirname(HERE), HERE]))
    p = subprocess.run([sys.executable, "-c", PRELUDE + body, host_hip, dtype], env=env, capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr


@pytest.mark.parametrize("dtype", ["f32", "int8"])
def test_finalize_after_a_failed_launch(host_hip, dtype):
    """Whichever launch of wgpt_model_finalize fails: the call fails, and a later one either has everything left as it needs it
    or is refused. After the first matrix was put into the order of the prefill products (the last 4 n_layer launches) the
    decode layouts can no longer be built from it."""
    run(host_hip, dtype, """
m = model()
at = launches.value
_lib.call("wgpt_model_finalize", m)
total, moves = launches.value - at, 4 * cfg["n_layer"]
assert total > moves
for i in range(1, total + 1):
    m = model()
    fail_at.value = launches.value + i
    assert refused("wgpt_model_finalize", m)
    fail_at.value = 0
    assert refused("wgpt_prefill", m, np.zeros(2, np.int32).ctypes.data_as(C.POINTER(C.c_int32)), 2, None)
    again = refused("wgpt_model_finalize", m)
    assert (again is not None) == (i > total - moves), (i, total, again)
    t = tensors["transformer.wpe.weight"]
    if again:
        assert "load the model again" in again
        assert refused("wgpt_model_set_tensor", m, b"transformer.wpe.weight", t.ctypes.data, t.nbytes)
    _lib.call("wgpt_model_destroy", m)
""")


def test_finalize_waits_for_its_launches(host_hip):
    """An error of the re-ordering belongs to wgpt_model_finalize, not to the first prefill: it returns with nothing in flight."""
    run(host_hip, "f32", """
m = model()
_lib.call("wgpt_model_finalize", m)
assert unwaited.value == 0, unwaited.value
""")


def test_finalize_after_a_failed_allocation(host_hip):
    """Whichever allocation of wgpt_model_finalize fails, a second call succeeds and the model runs."""
    run(host_hip, "f32", """
m = model()
at = allocs.value
_lib.call("wgpt_model_finalize", m)
total = allocs.value - at
tokens, logits = np.zeros(2, np.int32), np.zeros(cfg["vocab_size"], np.float32)
for i in range(1, total + 1):
    m = model()
    alloc_fail_at.value = allocs.value + i
    assert refused("wgpt_model_finalize", m)
    alloc_fail_at.value = 0
    _lib.call("wgpt_model_finalize", m)
    _lib.call("wgpt_prefill", m, tokens.ctypes.data_as(C.POINTER(C.c_int32)), 2, logits.ctypes.data_as(C.POINTER(C.c_float)))
    _lib.call("wgpt_decode_sample", m, 1, 2, 12, 1.0, np.zeros(2).ctypes.data_as(C.POINTER(C.c_double)), tokens.ctypes.data_as(C.POINTER(C.c_int32)), None)
    _lib.call("wgpt_model_destroy", m)
""")


@pytest.mark.parametrize("dtype", ["f32", "int8"])
def test_finalize_without_memory_for_the_pairs(host_hip, dtype):
    """Of a model whose products can be made of pairs of fp16 values: the one allocation of theirs may fail, and the model runs without them;
    behind every other failure a second call succeeds."""
    run(host_hip, dtype, """
cfg.update(n_embd=520, n_head=13, n_ctx=140, n_layer=1)
tensors = make_model(cfg, 1)
m = model()
at = allocs.value
_lib.call("wgpt_model_finalize", m)
total, without = allocs.value - at, 0
_lib.call("wgpt_model_destroy", m)
tokens = np.zeros(140, np.int32)
for i in range(1, total + 1):
    m = model()
    alloc_fail_at.value = allocs.value + i
    why = refused("wgpt_model_finalize", m)
    alloc_fail_at.value = 0
    without += why is None
    if why:
        assert refused("wgpt_model_finalize", m) is None, (i, why)
    for T in (140, 2):
        _lib.call("wgpt_prefill", m, tokens.ctypes.data_as(C.POINTER(C.c_int32)), T, None)
    _lib.call("wgpt_model_destroy", m)
assert without == 1, (without, total)
""")


@pytest.mark.parametrize("d,n_head,max_prefill,pairs", [(512, 8, 128, 0), (512, 8, 129, 1), (520, 13, 16, 1), (528, 4, 63, 0), (528, 4, 64, 1)])
def test_memory_of_the_pairs(host_hip, d, n_head, max_prefill, pairs):
    """A model whose prompts never read the pairs does not hold them: they all run in the persistent launch and on plain values (512 columns, 128
    tokens), or there is none (heads of 132) and they are too short."""
    run(host_hip, "f32", f"""
cfg.update(n_embd={d}, n_head={n_head}, n_ctx=140, n_layer=1)
made = []
for flags in (0, _lib.FLAG_TAPS):  # (with taps: no pairs)
    p = _lib.Params(**dict(synth.model_params(cfg)), max_prefill={max_prefill}, flags=flags)
    m = C.c_uint64(0)
    _lib.call("wgpt_model_create", C.byref(p), C.byref(m))
    for n, t in make_model(cfg, 1).items():
        _lib.call("wgpt_model_set_tensor", m, n.encode(), np.ascontiguousarray(t).ctypes.data, t.nbytes)
    at = allocs.value
    _lib.call("wgpt_model_finalize", m)
    made.append(allocs.value - at)
    _lib.call("wgpt_model_destroy", m)
assert made[0] - made[1] == {pairs}, made
""")


def test_buffers_of_a_window_that_grows(host_hip):
    """Nineteen buffers a window, given back behind it, as a forward from blocks has them: a window of a token more finds its memory among
    that of the shorter ones, also when those of many lengths have been left behind, and what is held stays within its bound."""
    run(host_hip, "f32", """
frees = C.c_int.in_dll(hip, "host_hip_frees")
own = allocs.value

def window(T, d=128):
    before = allocs.value
    hs = []
    for n in [d] * 12 + [4 * d] * 5 + [3 * d, 5003]:
        h = C.c_uint64(0)
        _lib.call("wgpt_alloc", 4 * T * n, C.byref(h))
        hs.append(h)
    for h in hs:
        _lib.call("wgpt_free", h)
    return allocs.value - before

assert [window(64) for _ in range(3)] == [19, 0, 0]
made = sum(window(T) for T in range(65, 1000))
assert made <= 19 * 16 * 4, made              # four octaves
assert sum(window(T) for T in range(900, 700, -1)) <= 19 * 8
big = [C.c_uint64(0) for _ in range(300)]      # a pass that does not fit keeps what it can
for _ in range(3):
    before = allocs.value
    for h in big:
        _lib.call("wgpt_alloc", 1 << 20, C.byref(h))
    made = allocs.value - before
    for h in big:
        _lib.call("wgpt_free", h)
assert made < 300 - 128, made
assert [window(10) for _ in range(60)][-1] == 0  # and makes room when nobody asks for it any more
assert allocs.value - frees.value - own <= 256, (allocs.value, frees.value)

# out of memory: what is kept is given back, then the size that was asked for is enough
h = C.c_uint64(0)
_lib.call("wgpt_shutdown")
_lib.init(0)
alloc_fail_at.value = allocs.value + 1
_lib.call("wgpt_alloc", 1000001, C.byref(h))   # nothing kept: a block of fewer bytes
size = C.c_size_t(0)
_lib.call("wgpt_buf_size", h, C.byref(size))
assert size.value == 1000001
_lib.call("wgpt_free", h)
before, alloc_fail_at.value = frees.value, allocs.value + 1
_lib.call("wgpt_alloc", 2000001, C.byref(h))
assert frees.value == before + 1
_lib.call("wgpt_free", h)
""")


@pytest.mark.parametrize("dtype", ["f32", "int8"])
def test_search_of_poll_delays_at_finalize(host_hip, dtype):
    """WGPT_FLAG_TUNE_DELAYS is for models whose context is long enough for a trial; the others load as they do without it."""
    run(host_hip, dtype, """
for ctx in (1, 2, 3, 4, 5, 24):
    cfg["n_ctx"] = ctx
    tensors = make_model(cfg, 1)
    p = _lib.Params(**synth.model_params(cfg), weight_dtype=int(sys.argv[2] == "int8"), flags=_lib.FLAG_TUNE_DELAYS)
    m = C.c_uint64(0)
    _lib.call("wgpt_model_create", C.byref(p), C.byref(m))
    for n, t in tensors.items():
        _lib.call("wgpt_model_set_tensor", m, n.encode(), np.ascontiguousarray(t).ctypes.data, t.nbytes)
    _lib.call("wgpt_model_finalize", m)
    again = refused("wgpt_model_tune_poll_delays", m, 0, None, None, None)
    assert (again is not None) == (ctx < 4) and (again is None or "context too short" in again), (ctx, again)
    _lib.call("wgpt_model_destroy", m)
""")
