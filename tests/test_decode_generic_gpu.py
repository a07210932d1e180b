"""Decode steps of shapes that the persistent kernel of fixed widths does not have (csrc/decode_generic.hip) against the CPU
oracle: widths of no whole segment, more heads than workgroups of a phase, head sizes up to 128, both weight dtypes, contexts on
both sides of the slices' limits, and what the host does when the launch gives up."""
import numpy as np
import pytest

from oracle import ref
from webgpt_amd import _lib, synth
from webgpt_amd._lib import WgptError
from webgpt_amd.model import GPT

from helpers import close, make_model, oracle_weights, pack_words, small_cfg, worst

pytestmark = pytest.mark.gpu

# (width, heads): the smallest, workgroups without columns (72), heads of 4, widths of no whole segment, one to seven segments
SHAPES = [(8, 1), (72, 2), (200, 5), (256, 64), (384, 32), (576, 12), (768, 8), (1032, 129), (1280, 10), (1600, 50), (1792, 14)]


def load(cfg, tensors):
    gpt = GPT(None, "char", tensors=tensors, params=synth.model_params(cfg))
    gpt.initialize()
    return gpt


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("d,n_head", SHAPES)
def test_steps_against_oracle_and_launches(device, dtype, d, n_head):
    """Single steps against the oracle and against a launch per block, from contexts around 64 and 128 positions (where a slice
    more is taken), then a run of greedy steps in one call; the rows that the steps leave in the cache."""
    cfg = small_cfg(n_layer=2, n_head=n_head, n_embd=d, n_ctx=200, vocab_size=301, dtype=dtype)
    tensors = make_model(cfg, d)
    gpt = load(cfg, tensors)
    gpt.set_decode_mode(1)
    w, p = oracle_weights(tensors, cfg), synth.model_params(cfg)
    tokens = synth.tokens(5, "prompt", 200, cfg["vocab_size"])
    for T in (1, 62, 127, 193):
        gpt.prefill(tokens[:T])
        for i in range(3):
            got = gpt.decode(int(tokens[T + i]))
            want, kv = ref.forward(p, w, tokens[:T + i + 1], want_kv=True)
            assert close(got, want), (T, i, worst(got, want))
        for li in range(2):
            for j, name in enumerate("kv"):
                rows = gpt.tap(f"kv{li}_{name}")
                assert close(rows, kv[li, j]), (T, li, name, worst(rows, kv[li, j]))
    assert gpt.routes()[1] == 1  # (no call was repeated with launches)
    out = {}
    for mode in (1, 0):
        gpt.set_decode_mode(mode)
        gpt.prefill(tokens[:60])
        out[mode] = gpt.decode_greedy(int(tokens[60]), 9, want_logits=True)
        assert gpt.routes()[1] == mode
    assert np.array_equal(out[1][0], out[0][0])
    assert close(out[1][1], out[0][1]), worst(out[1][1], out[0][1])
    gpt.unloadBuffers()


@pytest.mark.parametrize("n_head,n_embd,n_ctx", [(4, 512, 1024), (4, 256, 1024), (3, 96, 2048), (80, 1280, 1152)])
def test_the_longest_contexts(device, n_head, n_embd, n_ctx):
    """The last positions that the slices of a head hold in registers (heads of 128, 64 and 32; eighty heads in three slices)."""
    cfg = small_cfg(n_layer=1, n_head=n_head, n_embd=n_embd, n_ctx=n_ctx, vocab_size=97)
    tensors = make_model(cfg, 1)
    gpt = load(cfg, tensors)
    gpt.set_decode_mode(1)
    w, p = oracle_weights(tensors, cfg), synth.model_params(cfg)
    tokens = synth.tokens(3, "prompt", n_ctx, cfg["vocab_size"])
    for T in (509, n_ctx - 2):
        gpt.prefill(tokens[:T])
        for i in range(2):
            got = gpt.decode(int(tokens[T + i]))
            want = ref.forward(p, w, tokens[:T + i + 1])
            assert close(got, want), (T, i, worst(got, want))
    assert gpt.routes()[1] == 1
    gpt.unloadBuffers()


# vocabularies: fewer rows than workgroups, one row and some two, more than the 256 of a workgroup that registers hold
@pytest.mark.parametrize("vocab_size,repeat", [(5, 5), (301, 301), (301, 7), (5003, 5003), (70001, 70001), (70001, 3)])
def test_sampled_steps_select_what_the_oracle_selects(device, vocab_size, repeat):
    """Ids of sampled calls against the oracle's selection from the logits of single steps, whose arithmetic is the same; with a
    table of a few different rows the candidates are ties within and between workgroups, which the lowest index wins."""
    cfg = small_cfg(n_layer=1, n_head=2, n_embd=72, n_ctx=64, vocab_size=vocab_size)
    tensors = make_model(cfg, 2)
    wte = tensors["transformer.wte.weight"]
    tensors["transformer.wte.weight"] = np.ascontiguousarray(wte[np.arange(vocab_size) % repeat])
    gpt = load(cfg, tensors)
    gpt.set_decode_mode(1)
    tokens = synth.tokens(4, "prompt", 9, vocab_size)
    rng = np.random.default_rng(3)
    for top_k in (2, 3, 4, 5, 8):
        for steps in (1, 11):  # draws that travel with the launch, and in device memory
            u = rng.random(steps)
            gpt.prefill(tokens[:8])
            got = gpt.decode_sample(int(tokens[8]), steps, top_k, 0.8, u)
            gpt.prefill(tokens[:8])
            token = int(tokens[8])
            for i in range(steps):
                token = ref.sample_topk(gpt.decode(token), min(top_k, vocab_size), 0.8, float(u[i]))[0]
                assert token == got[i], (top_k, steps, i)
    assert gpt.routes()[1] == 1
    gpt.unloadBuffers()


@pytest.mark.parametrize("start", [2**31 - 1, 2**31 - 1 - 60, 2**31 - 1 - 200])
def test_epochs_restart_below_their_limit(device, monkeypatch, start):
    """The counter starts over, from cleared exchange buffers and both sets of candidates, in front of the first, the second or a later
    call: ids and logits of greedy and sampled calls are those of one from 0 on."""
    cfg = small_cfg(n_layer=2, n_head=4, n_embd=128, n_ctx=64, vocab_size=301)
    tensors, tokens, out = make_model(cfg, 3), synth.tokens(3, "prompt", 12, 301), []
    u = np.random.default_rng(3).random(5)
    for s in (0, start):
        monkeypatch.setenv("WEBGPT_AMD_EPOCH_START", str(s))
        gpt = load(cfg, tensors)
        gpt.set_decode_mode(1)
        gpt.prefill(tokens[:11])
        ids, rows = [int(tokens[11])], []
        for _ in range(4):
            more, last = gpt.decode_greedy(ids[-1], 4, want_logits=True)
            ids += [int(t) for t in more]
            rows.append(last)
            ids += [int(t) for t in gpt.decode_sample(ids[-1], 5, 8, 0.8, u)]
            rows.append(gpt.decode(ids[-1]))
        assert gpt.routes()[1] == 1
        out.append((ids, rows))
        gpt.unloadBuffers()
    assert out[0][0] == out[1][0] and all(np.array_equal(a, b) for a, b in zip(out[0][1], out[1][1]))


@pytest.mark.parametrize("dtype", ["f32", "int8"])
def test_expired_wait_repeats_the_call_with_launches(device, monkeypatch, dtype):
    """Waits that give up at their first look (forced from the host; every kernel drains): the calls succeed with the results of a
    launch per block, bit for bit."""
    cfg = small_cfg(n_layer=2, n_head=4, n_embd=128, n_ctx=64, vocab_size=90, dtype=dtype)
    tensors = make_model(cfg, 3)
    monkeypatch.setenv("WEBGPT_AMD_SPIN_LIMIT", "0")
    monkeypatch.setenv("WEBGPT_AMD_POLL_DELAYS", "0,0,0,0,0,0,0")
    launches = load(cfg, tensors)  # (its prompts give up as well: the caches are the same)
    launches.set_decode_mode(0)
    tokens = synth.tokens(9, "prompt", 20, cfg["vocab_size"])
    u = np.array([0.3, 0.6, 0.9])
    calls = [lambda g: g.decode(int(tokens[12])), lambda g: g.decode_greedy(int(tokens[12]), 3), lambda g: g.decode_sample(int(tokens[12]), 3, 5, 0.8, u)]
    for call in calls:
        gpt = load(cfg, tensors)
        for g in (gpt, launches):
            g.prefill(tokens[:12])
        assert np.array_equal(call(gpt), call(launches))
        assert gpt.routes() == (0, 0)
        assert np.array_equal(gpt.decode(int(tokens[16])), launches.decode(int(tokens[16])))
        with pytest.raises(WgptError, match="not available"):
            gpt.set_decode_mode(1)
        gpt.unloadBuffers()
    launches.unloadBuffers()


@pytest.mark.parametrize("dtype", ["f32", "int8"])
def test_rows_whose_variance_overflows(device, dtype):
    """Finite residual values of 1e28: a row's variance is infinite, its quotients are zeros and the LayerNorm's result is beta."""
    cfg = small_cfg(n_layer=2, n_head=5, n_embd=200, n_ctx=64, vocab_size=90, dtype=dtype)
    tensors = make_model(cfg, 5)
    tensors["transformer.wpe.weight"] = tensors["transformer.wpe.weight"] * np.float32(1e30)
    gpt = load(cfg, tensors)
    gpt.set_decode_mode(1)
    w, p = oracle_weights(tensors, cfg), synth.model_params(cfg)
    tokens = synth.tokens(5, "prompt", 20, cfg["vocab_size"])
    with np.errstate(all="ignore"):
        gpt.prefill(tokens[:17])
        for i in range(17, 20):
            got, want = gpt.decode(int(tokens[i])), ref.forward(p, w, tokens[:i + 1])
            assert np.isfinite(want).all() and close(got, want), i
    assert gpt.routes()[1] == 1
    gpt.unloadBuffers()


@pytest.mark.parametrize("dtype", ["f32", "int8"])
def test_rows_of_one_huge_value(device, dtype):
    """All elements of a row 2^120: its LayerNorm is beta, at a width that leaves lanes without elements, whose zeros are 2^128 standard
    deviations from the mean."""
    cfg = small_cfg(n_layer=2, n_head=2, n_embd=40, n_ctx=64, vocab_size=90, dtype=dtype)
    tensors = make_model(cfg, 5)
    tensors["transformer.wpe.weight"] = np.full_like(tensors["transformer.wpe.weight"], 2.0 ** 120)
    gpt = load(cfg, tensors)
    w, p = oracle_weights(tensors, cfg), synth.model_params(cfg)
    gpt.set_decode_mode(1)
    tokens = synth.tokens(5, "prompt", 20, cfg["vocab_size"])
    gpt.prefill(tokens[:17])
    for i in range(17, 20):
        got, want = gpt.decode(int(tokens[i])), ref.forward(p, w, tokens[:i + 1])
        assert np.isfinite(want).all() and close(got, want), i
    assert gpt.routes()[1] == 1
    gpt.unloadBuffers()


@pytest.mark.parametrize("inputs,product", [("ln_1.bias", "attn.c_attn"), ("attn.c_attn.bias", "attn.c_proj"), ("ln_2.bias", "mlp.c_fc"), ("mlp.c_fc.bias", "mlp.c_proj")])
def test_int8_sums_beyond_the_range_of_fp32(device, inputs, product):
    """Inputs of 1e35 in front of one product, whose column scales bring its results back to about 1e2: the sums of 127 x 1e35 and less are infinite
    before the scale meets them. Of c_attn only the values' columns (the scores stay small)."""
    d = 200
    cfg = small_cfg(n_layer=2, n_head=5, n_embd=d, n_ctx=64, vocab_size=90, dtype="int8")
    tensors = make_model(cfg, 5)
    p, rng = "transformer.h.0.", np.random.default_rng(3)
    K, N = (4 * d if product == "mlp.c_proj" else d), {"attn.c_attn": 3 * d, "mlp.c_fc": 4 * d}.get(product, d)
    q, scale = rng.integers(1, 128, (K, N)).astype(np.int8), np.full(N, 127e-37, np.float32)
    if product == "attn.c_attn":
        q[:, :2 * d] = 0
    tensors[p + inputs] = np.full_like(tensors[p + inputs], 1e35)
    if inputs == "attn.c_attn.bias":
        tensors[p + inputs][:2 * d] = 0
    tensors[p + product + ".weight.q"], tensors[p + product + ".weight.scale"] = pack_words(q), scale
    gpt = load(cfg, tensors)
    gpt.set_decode_mode(1)
    w, prm = oracle_weights(tensors, cfg), synth.model_params(cfg)
    tokens = synth.tokens(5, "prompt", 20, cfg["vocab_size"])
    gpt.prefill(tokens[:17])
    for i in range(17, 20):
        got, want = gpt.decode(int(tokens[i])), ref.forward(prm, w, tokens[:i + 1])
        assert np.isfinite(want).all() and close(got, want), (i, worst(got, want))
    assert gpt.routes()[1] == 1
    gpt.unloadBuffers()


def test_expired_wait_in_a_search_of_delays(device, monkeypatch):
    """A search whose trials give up says so; where it is a part of loading the model, the model is loaded. Both decode with launches."""
    cfg = small_cfg(n_layer=2, n_head=4, n_embd=128, n_ctx=64, vocab_size=90)
    tensors = make_model(cfg, 3)
    monkeypatch.setenv("WEBGPT_AMD_SPIN_LIMIT", "0")
    monkeypatch.setenv("WEBGPT_AMD_POLL_DELAYS", "0,0,0,0,0,0,0")
    tokens, rows = synth.tokens(9, "prompt", 20, cfg["vocab_size"]), []
    for flags in (0, _lib.FLAG_TUNE_DELAYS):
        gpt = GPT(None, "char", tensors=tensors, params=synth.model_params(cfg), flags=flags)
        gpt.initialize()
        if not flags:
            with pytest.raises(WgptError, match="a wait of a trial launch expired"):
                gpt.tune_poll_delays(1)
        with pytest.raises(WgptError, match="not available"):
            gpt.set_decode_mode(1)
        gpt.prefill(tokens[:12])
        rows.append(gpt.decode(int(tokens[12])))
        gpt.unloadBuffers()
    assert np.array_equal(rows[0], rows[1])
    assert close(rows[0], ref.forward(synth.model_params(cfg), oracle_weights(tensors, cfg), tokens[:13]))


@pytest.mark.parametrize("vocab_size", [301, 5003])
def test_logits_that_are_no_numbers_hide_no_others(device, vocab_size):
    """Every second token's embedding is NaN, and so is its logit: greedy steps choose among the others, as the selection for sampling does."""
    cfg = small_cfg(n_layer=2, n_head=4, n_embd=128, n_ctx=64, vocab_size=vocab_size)
    tensors = make_model(cfg, 3)
    wte = tensors["transformer.wte.weight"].copy()
    wte[2::2] = np.nan
    tensors["transformer.wte.weight"] = wte
    gpt = load(cfg, tensors)
    gpt.set_decode_mode(1)
    w, p = oracle_weights(tensors, cfg), synth.model_params(cfg)
    history = [int(t) // 2 * 2 - 1 for t in synth.tokens(9, "prompt", 12, vocab_size) if t > 1]
    gpt.prefill(history[:-1])
    got = [int(t) for t in gpt.decode_greedy(history[-1], 4)]
    gpt.prefill(history[:-1])
    sampled = [int(t) for t in gpt.decode_sample(history[-1], 4, 1, 0.8, np.full(4, 0.5))]
    assert gpt.routes()[1] == 1
    with np.errstate(all="ignore"):
        for t in got:
            assert t == int(np.nanargmax(ref.forward(p, w, np.array(history, np.int32))))
            history.append(t)
    assert sampled == got
    gpt.unloadBuffers()
