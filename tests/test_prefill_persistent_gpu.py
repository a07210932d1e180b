"""Prompts that run as one persistent launch (wgpt_prefill, csrc/prefill_persistent.hip) against the CPU oracle: edges of the
sixteen rows of a row group, of the steps of 32 of a contraction and of the tiles of sixteen columns, head sizes, both weight
dtypes, and what the host does when the launch gives up."""
import numpy as np
import pytest

from oracle import ref
from webgpt_amd import _lib, blocks, synth
from webgpt_amd.model import GPT

from helpers import close, make_model, oracle_weights, pack_words, small_cfg, worst

pytestmark = pytest.mark.gpu

# (width, heads): the smallest, widths of no whole step or slice, more heads than column groups, head sizes up to 128, the widest
SHAPES = [(8, 1), (40, 2), (200, 5), (256, 2), (576, 12), (640, 40), (1240, 31), (1280, 10), (1600, 25), (1792, 14)]


def load(cfg, tensors, flags=0):
    gpt = GPT(None, "char", tensors=tensors, params=synth.model_params(cfg), flags=flags)
    gpt.initialize()
    return gpt


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("d,n_head", SHAPES)
def test_prompts_against_oracle(device, dtype, d, n_head):
    """Logits, cache rows of both layers and the residual rows, of one model in turn: a launch meets what the one before it left."""
    cfg = small_cfg(n_layer=2, n_head=n_head, n_embd=d, n_ctx=130, vocab_size=301, dtype=dtype)
    tensors = make_model(cfg, d)
    gpt = load(cfg, tensors)
    w, p = oracle_weights(tensors, cfg), synth.model_params(cfg)
    for T in (1, 16, 128, 17, 2, 61, 64, 65, 113, 129):
        tokens = synth.tokens(T, "prompt", T, cfg["vocab_size"])
        want, taps, kv = ref.forward(p, w, tokens, want_taps=True, want_kv=True)
        got = gpt.prefill(tokens)
        assert close(got, want), (T, worst(got, want))
        assert gpt.routes()[0] == (T <= (64 if dtype == "f32" and d > 1280 else 128)), T
        for i in range(2):
            for j, name in enumerate("kv"):
                rows = gpt.tap(f"kv{i}_{name}")
                assert close(rows, kv[i, j]), (T, i, name, worst(rows, kv[i, j]))
        # a residual value is the sum of an embedding and four products of the rows' size: near zero its error is that of its
        # terms (d = 1600: 1e-5 of their root mean square, of which the oracle's ascending fp32 sums have the larger half)
        rows, exp = gpt.tap("residual", T), taps[ref.tap_names(2).index("block1_r2")]
        assert close(rows, exp, atol=1e-4 * float(np.sqrt(np.mean(exp ** 2)))), T
    gpt.unloadBuffers()


def test_memory_as_it_was_left(device):
    """A model in memory full of NaN, as far as the driver hands out again what was given back to it (the library keeps no buffers that
    the host has written to): what the row group's rows beyond the prompt hold does not end the launch, and the logits are those of the same
    model in other memory, bit for bit. (Rows that an earlier prompt has left there for certain:
    test_a_spoilt_prompt_is_no_matter_of_the_next_ones.)"""
    cfg = small_cfg(n_layer=2, n_head=4, n_embd=256, n_ctx=64, vocab_size=301, dtype="int8")
    tensors, tokens = make_model(cfg, 5), synth.tokens(5, "prompt", 16, cfg["vocab_size"])

    def run():
        gpt = load(cfg, tensors)
        got = []
        for T in (13, 16, 1):
            got.append(gpt.prefill(tokens[:T]))
            assert gpt.routes()[0] == 1, T
        gpt.unloadBuffers()
        return got

    want = run()
    nan = np.full(8 << 20, np.nan, np.float32)
    junk = [blocks.init_tensor(nan, [nan.size]) for _ in range(16)]
    for b in junk:
        b.destroy()
    for a, b in zip(want, run()):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("dtype", ["f32", "int8"])
def test_expired_wait_falls_back_to_launches(device, monkeypatch, dtype):
    """Waits that give up at their first look (forced from the host; every kernel drains): the call's results are those of the
    launches, to which every later call goes at once, bit for bit."""
    cfg = small_cfg(n_layer=2, n_head=4, n_embd=128, n_ctx=64, vocab_size=90, dtype=dtype)
    tensors = make_model(cfg, 3)
    launches = load(cfg, tensors, flags=_lib.FLAG_TAPS)  # (with taps a prompt always takes them)
    monkeypatch.setenv("WEBGPT_AMD_SPIN_LIMIT", "0")
    gpt = load(cfg, tensors)
    monkeypatch.delenv("WEBGPT_AMD_SPIN_LIMIT")
    w, p = oracle_weights(tensors, cfg), synth.model_params(cfg)
    for T in (40, 12):
        tokens = synth.tokens(T, "prompt", T, cfg["vocab_size"])
        got = gpt.prefill(tokens)
        assert gpt.routes()[0] == 0 and close(got, ref.forward(p, w, tokens)) and close(got, launches.prefill(tokens)), T
        assert np.array_equal(got, gpt.prefill(tokens)), T
    gpt.unloadBuffers()
    launches.unloadBuffers()


@pytest.mark.parametrize("start", [2**31 - 1, 2**31 - 1 - 22, 2**31 - 1 - 33])
def test_epochs_restart_below_their_limit(device, monkeypatch, start):
    """Eleven epochs a prompt: the counter starts over in front of the first, second or third prompt, with the bits of one from 0 on."""
    cfg = small_cfg(n_layer=2, n_head=4, n_embd=128, n_ctx=64, vocab_size=90)
    tensors, tokens, rows = make_model(cfg, 3), synth.tokens(3, "prompt", 64, 90), []
    for s in (0, start):
        monkeypatch.setenv("WEBGPT_AMD_EPOCH_START", str(s))
        gpt = load(cfg, tensors)
        rows.append([gpt.prefill(tokens[:T]) for T in (40, 64, 12, 33, 64)])
        assert gpt.routes()[0] == 1
        gpt.unloadBuffers()
    assert all(np.array_equal(a, b) for a, b in zip(*rows))


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("what", ["value", "scale", "weight"])
def test_values_that_are_not_finite(device, dtype, what):
    """A bias of the values that is infinite, an infinite column scale (int8) or weight (fp32), tiny embeddings: rows that the
    launches lose are lost and all others as they give them."""
    cfg = small_cfg(n_layer=2, n_head=4, n_embd=128, n_ctx=64, vocab_size=90, dtype=dtype)
    tensors = make_model(cfg, 5)
    T = 50
    tokens = synth.tokens(T, "prompt", T, cfg["vocab_size"])
    if what == "value":  # one position's embedding: its keys and values are NaN, queries before it must not see them
        tensors["transformer.wpe.weight"] = tensors["transformer.wpe.weight"].copy()
        tensors["transformer.wpe.weight"][37, 5] = np.inf
    else:
        name = "transformer.h.1.mlp.c_fc." + ("weight" if dtype == "f32" else "weight.scale")
        if what == "weight":
            name = "transformer.wpe.weight"  # products of nothing but tiny values behind a LayerNorm that divides by sqrt(1e-5)
            tensors["transformer.wte.weight"] = tensors["transformer.wte.weight"] * np.float32(0)
            tensors[name] = tensors[name] * np.float32(1e-30)
        else:
            tensors[name] = tensors[name].copy()
            tensors[name].reshape(-1)[7] = np.inf
    launches = load(cfg, tensors, flags=_lib.FLAG_TAPS)
    gpt = load(cfg, tensors)
    with np.errstate(all="ignore"):
        got, want = gpt.prefill(tokens), launches.prefill(tokens)
        for i in range(2):
            for name in "kv":
                a, b = gpt.tap(f"kv{i}_{name}"), launches.tap(f"kv{i}_{name}")
                assert (np.isfinite(a) == np.isfinite(b)).all(), (i, name)
                ok = np.isfinite(b)
                assert close(a[ok], b[ok]), (i, name)
        assert (np.isfinite(got) == np.isfinite(want)).all()
        ok = np.isfinite(want)
        assert close(got[ok], want[ok])
    gpt.unloadBuffers()
    launches.unloadBuffers()


@pytest.mark.parametrize("dtype", ["f32", "int8"])
def test_a_spoilt_prompt_is_no_matter_of_the_next_ones(device, dtype):
    """Prompts before and behind one with a value that is not finite: the same bits (launches round in another order), also where the row
    group holds rows that the spoilt one has left. Behind several spoilt ones prompts are tried again after a while."""
    cfg = small_cfg(n_layer=2, n_head=4, n_embd=128, n_ctx=64, vocab_size=90, dtype=dtype)
    tensors = make_model(cfg, 5)
    tensors["transformer.wpe.weight"] = tensors["transformer.wpe.weight"].copy()
    tensors["transformer.wpe.weight"][37, 5] = np.inf
    tokens = synth.tokens(5, "prompt", 50, cfg["vocab_size"])
    gpt = load(cfg, tensors)
    lengths = (35, 12, 37, 1)
    alone = {T: gpt.prefill(tokens[:T]) for T in lengths}
    with np.errstate(all="ignore"):
        for T in lengths:
            gpt.prefill(tokens)
            assert gpt.routes()[0] == 0
            for again in lengths[:lengths.index(T) + 1]:
                assert np.array_equal(gpt.prefill(tokens[:again]), alone[again]) and gpt.routes()[0] == 1, (T, again)
        for _ in range(5):
            gpt.prefill(tokens)
        got = [gpt.prefill(tokens[:35]) for _ in range(8)]
    assert all(close(g, alone[35]) for g in got) and np.array_equal(got[-1], alone[35]) and gpt.routes()[0] == 1
    gpt.unloadBuffers()


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("name", ["wpe.weight", "h.1.attn.c_proj.bias", "h.1.mlp.c_proj.bias"])
def test_rows_whose_variance_overflows(device, dtype, name):
    """Finite residual values of 1e28 from the first, the last and the final LayerNorm on: a row's variance is infinite, its quotients
    are zeros and the LayerNorm's result is beta."""
    cfg = small_cfg(n_layer=2, n_head=5, n_embd=200, n_ctx=64, vocab_size=90, dtype=dtype)
    tensors = make_model(cfg, 5)
    tensors["transformer." + name] = tensors["transformer." + name] * np.float32(1e30)
    gpt = load(cfg, tensors)
    w, p = oracle_weights(tensors, cfg), synth.model_params(cfg)
    for T in (1, 20, 64):
        tokens = synth.tokens(T, "prompt", T, cfg["vocab_size"])
        with np.errstate(all="ignore"):
            got, want = gpt.prefill(tokens), ref.forward(p, w, tokens)
        assert np.isfinite(want).all() and close(got, want) and gpt.routes()[0] == 1, T
    gpt.unloadBuffers()


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("n_head", [1, 4])
def test_sixteen_keys_whose_scores_overflow(device, dtype, n_head):
    """Scores of minus infinity for all keys of the first row group, whose weights are then zero, and finite ones for all others:
    a LayerNorm that passes the sign of the first sixteen rows' first element and zeros for the others, keys that are 1e20 of it."""
    d, T = 64, 40
    cfg = small_cfg(n_layer=1, n_head=n_head, n_embd=d, n_ctx=64, vocab_size=90, dtype=dtype)
    tensors = make_model(cfg, 5)
    wte, wpe = np.zeros((90, d), np.float32), np.zeros((64, d), np.float32)
    wte[:, 3] = np.arange(90)  # (token 0, which the prompt repeats, has no embedding)
    wpe[:16, 0], wpe[:16, 1] = 1, -1
    tensors.update({"transformer.wte.weight": wte, "transformer.wpe.weight": wpe, "transformer.h.0.ln_1.bias": np.zeros(d, np.float32)})
    bias = tensors["transformer.h.0.attn.c_attn.bias"].copy()
    bias[:d], bias[d:2 * d] = -1e20, 0
    tensors["transformer.h.0.attn.c_attn.bias"] = bias
    name = "transformer.h.0.attn.c_attn.weight"
    if dtype == "f32":
        W = tensors[name].copy()
        W[:, :2 * d] = 0
        W[0, d:2 * d] = 1e20
        tensors[name] = W
    else:
        q = np.random.default_rng(3).integers(-127, 128, (d, 3 * d)).astype(np.int8)
        q[:, :2 * d] = 0
        q[0, d:2 * d] = 127
        tensors[name + ".q"] = pack_words(q)
        scale = tensors[name + ".scale"].copy()
        scale[d:2 * d] = 1e20
        tensors[name + ".scale"] = scale
    gpt = load(cfg, tensors)
    w, p = oracle_weights(tensors, cfg), synth.model_params(cfg)
    tokens = np.zeros(T, np.int32)
    with np.errstate(all="ignore"):
        got, want = gpt.prefill(tokens), ref.forward(p, w, tokens)
    assert np.isfinite(want).all() and close(got, want), worst(got, want)
    assert dtype == "int8" or gpt.routes()[0] == 1
    gpt.unloadBuffers()


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("name", ["wpe.weight", "h.1.attn.c_proj.bias"])
def test_rows_of_one_huge_value(device, dtype, name):
    """All elements of a row 2^120: its LayerNorm is beta, at a width that leaves lanes without elements, whose zeros are 2^128 standard
    deviations from the mean."""
    cfg = small_cfg(n_layer=2, n_head=2, n_embd=40, n_ctx=64, vocab_size=90, dtype=dtype)
    tensors = make_model(cfg, 5)
    tensors["transformer." + name] = np.full_like(tensors["transformer." + name], 2.0 ** 120)
    gpt = load(cfg, tensors)
    w, p = oracle_weights(tensors, cfg), synth.model_params(cfg)
    for T in (1, 20, 64):
        tokens = synth.tokens(T, "prompt", T, cfg["vocab_size"])
        got, want = gpt.prefill(tokens), ref.forward(p, w, tokens)
        assert np.isfinite(want).all() and close(got, want) and gpt.routes()[0] == 1, T
    gpt.unloadBuffers()
