"""Longer prompts, whose products are made of pairs of fp16 values (csrc/gemm_pair.hip), against the CPU oracle: edges of the tiles'
rows and columns, widths of no whole run of sixteen, both weight dtypes, and models whose weights the pairs cannot take."""
import numpy as np
import pytest

from oracle import ref
from webgpt_amd import _lib, synth
from webgpt_amd.model import GPT

from helpers import close, make_model, oracle_weights, small_cfg, worst

pytestmark = pytest.mark.gpu

FLAG_TAPS = 1


def load(cfg, tensors, flags=0):
    gpt = GPT(None, "char", tensors=tensors, params=synth.model_params(cfg), flags=flags)
    gpt.initialize()
    return gpt


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("d,n_head", [(512, 8), (520, 13), (576, 12), (1288, 23), (1608, 67)])
def test_prompts_against_oracle(device, dtype, d, n_head):
    """Logits, cache rows and residual rows, of one model in turn: a longer prompt's rows are left behind a shorter one's. Widths of
    sixteen and of eight, heads of 64, 40, 48, 56 and 24. A model that keeps taps runs the other products: other last bits."""
    cfg = small_cfg(n_layer=2, n_head=n_head, n_embd=d, n_ctx=260, vocab_size=301, dtype=dtype)
    tensors = make_model(cfg, d)
    gpt, taps = load(cfg, tensors), load(cfg, tensors, FLAG_TAPS)
    w, p = oracle_weights(tensors, cfg), synth.model_params(cfg)
    for T in (129, 257, 160, 193, 161, 192):
        tokens = synth.tokens(T, "prompt", T, cfg["vocab_size"])
        want, all_taps, kv = ref.forward(p, w, tokens, want_taps=True, want_kv=True)
        got = gpt.prefill(tokens)
        assert close(got, want), (T, worst(got, want))
        assert not np.array_equal(got, taps.prefill(tokens)), T
        assert gpt.pairs() == 1 and taps.pairs() == 0, T
        for i in range(2):
            for j, name in enumerate("kv"):
                assert close(gpt.tap(f"kv{i}_{name}"), kv[i, j]), (T, i, name)
        rows, exp = gpt.tap("residual", T), all_taps[ref.tap_names(2).index("block1_r2")]
        # (a sum of five values of the rows' size: near zero its error is theirs)
        assert close(rows, exp, atol=1e-4 * float(np.sqrt(np.mean(exp ** 2)))), T
    gpt.unloadBuffers()
    taps.unloadBuffers()


def spoil(tensors, how):
    name = "transformer.h.1.mlp.c_fc.weight"
    t = {k: v.copy() for k, v in tensors.items()}
    if how == "infinite":
        t[name][3, 5] = np.inf
    elif how == "tiny columns":  # all but one weight of a column 2^-30 of that one
        t[name][1:, 7] *= np.float32(2.0 ** -30)
    elif how == "tiny":
        t[name] *= np.float32(2.0 ** -100)
    elif how == "gamma":
        t["transformer.h.0.ln_2.weight"][1:] *= np.float32(2.0 ** -20)
    elif how == "large":  # a bound beyond what the rows' scales reach
        t["transformer.h.1.mlp.c_fc.bias"][0] = 2.0 ** 70
    return t


@pytest.mark.parametrize("how", ["infinite", "tiny columns", "tiny", "gamma", "large"])
def test_weights_beyond_the_pairs(device, how):
    """Found when the model is loaded, which then runs the products of a model that keeps taps."""
    cfg = small_cfg(n_layer=2, n_head=8, n_embd=512, n_ctx=140, vocab_size=101)
    tensors = spoil(make_model(cfg, 3), how)
    tokens = synth.tokens(3, "prompt", 140, cfg["vocab_size"])
    gpt, taps = load(cfg, tensors), load(cfg, tensors, FLAG_TAPS)
    got, want = gpt.prefill(tokens), taps.prefill(tokens)
    assert gpt.pairs() == 0
    # (the LayerNorm in front of a product is a pass of its own where there are taps: equal to rounding, not to the last bit)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and close(got[~np.isnan(want)], want[~np.isnan(want)])
    gpt.unloadBuffers()
    taps.unloadBuffers()


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("d,n_head,T", [(512, 8, 140), (520, 13, 140), (520, 13, 60), (1024, 16, 60)])
@pytest.mark.parametrize("how", ["dead unit", "value column", "value head", "ln_1 beta", "ln_2 beta", "ln_2 gamma"])
def test_one_wide_column(device, dtype, d, n_head, T, how):
    """A bound far beyond the others', in the rows that a product reads: what the others' values hold is not lost. A hidden unit that its
    bias keeps at zero; values that c_proj's rows make up for; a channel of a LayerNorm that nothing reads."""
    cfg = small_cfg(n_layer=2, n_head=n_head, n_embd=d, n_ctx=140, vocab_size=101, dtype=dtype)
    tensors = {k: v.copy() for k, v in make_model(cfg, 3).items()}
    p = "transformer.h.1."
    if how == "dead unit":
        tensors[p + "mlp.c_fc.bias"][0] = -1e9
    elif how.startswith("ln"):
        reader = "attn.c_attn.weight" if how.startswith("ln_1") else "mlp.c_fc.weight"
        tensors[p + how[:4] + (".bias" if how.endswith("beta") else ".weight")][0] = 1e9
        tensors[p + reader + (".q" if dtype == "int8" else "")][0] = 0
    else:
        cols, up = slice(2 * d + 3, 2 * d + 4) if how == "value column" else slice(2 * d, 2 * d + d // n_head), 24
        rows = slice(cols.start - 2 * d, cols.stop - 2 * d)
        tensors[p + "attn.c_attn.bias"][cols] *= np.float32(2.0 ** up)
        if dtype == "f32":
            tensors[p + "attn.c_attn.weight"][:, cols] *= np.float32(2.0 ** up)
            tensors[p + "attn.c_proj.weight"][rows] *= np.float32(2.0 ** -up)
        else:  # (no row of int8 weights is that small: without the column)
            tensors[p + "attn.c_attn.weight.scale"][cols] *= np.float32(2.0 ** up)
            tensors[p + "attn.c_proj.weight.q"][rows] = 0
    gpt, tokens = load(cfg, tensors), synth.tokens(3, "prompt", T, cfg["vocab_size"])
    want = ref.forward(synth.model_params(cfg), oracle_weights(tensors, cfg), tokens)
    got = gpt.prefill(tokens)
    assert close(got, want), worst(got, want)
    assert gpt.pairs() == 0
    gpt.unloadBuffers()


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("d,n_head,rows", [(1608, 67, (513, 401, 400)), (1600, 25, (513, 400))])
def test_many_rows_of_wide_models(device, dtype, d, n_head, rows):
    """Both sides of the rule for the LayerNorm's workgroups (a row each up to 400 rows) at widths beyond three runs of 512."""
    cfg = small_cfg(n_layer=1, n_head=n_head, n_embd=d, n_ctx=520, vocab_size=97, dtype=dtype)
    tensors = make_model(cfg, d)
    gpt, w, p = load(cfg, tensors), oracle_weights(tensors, cfg), synth.model_params(cfg)
    for T in rows:
        tokens = synth.tokens(T, "prompt", T, cfg["vocab_size"])
        want, taps, _ = ref.forward(p, w, tokens, want_taps=True, want_kv=True)
        got = gpt.prefill(tokens)
        assert close(got, want) and gpt.pairs() == 1, (T, worst(got, want))
        rows_got, exp = gpt.tap("residual", T), taps[ref.tap_names(1).index("block0_r2")]
        assert close(rows_got, exp, atol=1e-4 * float(np.sqrt(np.mean(exp ** 2)))), T  # (near zero a sum's error is its terms')
    gpt.unloadBuffers()


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("d,n_head,rows", [(768, 12, (961, 960, 943, 865)), (744, 6, (513, 385, 289)), (1000, 10, (300, 193)), (1600, 25, (300, 129)),
                                           (1240, 31, (943, 300)), (2056, 257, (513,)), (512, 8, (257, 140))])
def test_prompts_without_the_pairs(device, dtype, d, n_head, rows):
    """A gain that the pairs' scale does not fit: products of three bf16 values each, LayerNorm, GELU and cache rows with them, at the edges of
    their larger tiles."""
    cfg = small_cfg(n_layer=1, n_head=n_head, n_embd=d, n_ctx=1024, vocab_size=97, dtype=dtype)
    tensors = {k: v.copy() for k, v in make_model(cfg, d).items()}
    tensors["transformer.h.0.ln_2.weight"][3] = 2.0 ** -20
    tensors["transformer.h.0.ln_2.bias"][3] = 0.0
    gpt, w, p = load(cfg, tensors), oracle_weights(tensors, cfg), synth.model_params(cfg)
    for T in rows:
        tokens = synth.tokens(T, "prompt", T, cfg["vocab_size"])
        want, taps, kv = ref.forward(p, w, tokens, want_taps=True, want_kv=True)
        got = gpt.prefill(tokens)
        assert close(got, want) and gpt.pairs() == 0, (T, worst(got, want))
        for j, name in enumerate("kv"):
            assert close(gpt.tap(f"kv0_{name}"), kv[0, j]), (T, name)
        rows_got, exp = gpt.tap("residual", T), taps[ref.tap_names(1).index("block0_r2")]
        assert close(rows_got, exp, atol=1e-4 * float(np.sqrt(np.mean(exp ** 2)))), T  # (near zero a sum's error is its terms')
    gpt.unloadBuffers()


def test_rows_that_are_no_numbers(device):
    """An embedding that is infinite makes its row's logits and those of the rows behind it NaN, and none of the tiles before it; the next
    prompt is not affected by what was left in the rows' memory."""
    cfg = small_cfg(n_layer=2, n_head=8, n_embd=512, n_ctx=300, vocab_size=101)
    tensors = make_model(cfg, 4)
    clean = load(cfg, tensors)
    bad = {k: v.copy() for k, v in tensors.items()}
    bad["transformer.wte.weight"][100, 9] = np.inf
    gpt = load(cfg, bad)
    tokens = [int(t) % 100 for t in synth.tokens(4, "prompt", 299, cfg["vocab_size"])]
    spoilt = list(tokens)
    spoilt[150] = 100
    want = clean.prefill(tokens[:200])[:100]
    assert np.isnan(gpt.prefill(spoilt)[:100]).all()
    assert np.isnan(gpt.tap("residual", 299)[151:]).any(axis=1).all() and np.isfinite(gpt.tap("residual", 299)[:128]).all()
    for T in (200, 150):
        got = gpt.prefill(tokens[:T])[:100]
        assert np.isfinite(got).all() and np.array_equal(got, clean.prefill(tokens[:T])[:100])
    assert np.array_equal(gpt.prefill(tokens[:200])[:100], want)
    gpt.unloadBuffers()
    clean.unloadBuffers()


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("d,n_head", [(512, 8), (768, 12), (640, 5)])
def test_shorter_prompt_behind_a_longer_one(device, dtype, d, n_head):
    """A gain of 64 that c_attn's row makes up for: the rows that the longer prompt's last layer left behind are far beyond what the first
    one's values can be, and the shorter prompt has the results of a fresh model."""
    cfg = small_cfg(n_layer=2, n_head=n_head, n_embd=d, n_ctx=300, vocab_size=301, dtype=dtype)
    tensors = {k: v.copy() for k, v in make_model(cfg, 6).items()}
    for i in range(2):
        p = f"transformer.h.{i}."
        tensors[p + "ln_1.weight"][5] = 64.0
        if dtype == "f32":
            tensors[p + "attn.c_attn.weight"][5] /= 64.0
        else:
            tensors[p + "attn.c_attn.weight.q"][5] = 0x01FF01FF  # (-1, 1, -1, 1)
    tokens = synth.tokens(7, "prompt", 300, cfg["vocab_size"])
    fresh, gpt = load(cfg, tensors), load(cfg, tensors)
    w, p = oracle_weights(tensors, cfg), synth.model_params(cfg)
    gpt.prefill(tokens)
    for T in (150, 131):
        want, got = fresh.prefill(tokens[:T]), gpt.prefill(tokens[:T])
        assert np.array_equal(got, want) and close(got, ref.forward(p, w, tokens[:T])), T
        assert gpt.pairs() == 1, T
        gpt.prefill(tokens)
        fresh.unloadBuffers()
        fresh = load(cfg, tensors)
    gpt.unloadBuffers()
    fresh.unloadBuffers()


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("d,n_head", [(520, 13), (1024, 16), (1288, 23), (1608, 67)])
def test_short_prompts_of_weights_beyond_the_pairs(device, dtype, d, n_head):
    """One column that the pairs cannot take: short prompts run in one launch all the same, on plain values."""
    cfg = small_cfg(n_layer=2, n_head=n_head, n_embd=d, n_ctx=70, vocab_size=101, dtype=dtype)
    tensors = spoil(make_model(cfg, 8), "tiny columns") if dtype == "f32" else make_model(cfg, 8)
    if dtype == "int8":
        name = "transformer.h.1.mlp.c_fc.weight.scale"
        tensors[name] = tensors[name].copy()
        tensors[name][7] = 2.0 ** -100
    gpt, w, p = load(cfg, tensors), oracle_weights(tensors, cfg), synth.model_params(cfg)
    for T in (1, 17, 61):
        tokens = synth.tokens(T, "prompt", T, cfg["vocab_size"])
        want = ref.forward(p, w, tokens)
        got = gpt.prefill(tokens)
        assert close(got, want), (T, worst(got, want))
        assert gpt.routes()[0] == 1 and gpt.pairs() == 0, T
    gpt.unloadBuffers()


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("d,n_head,pairs", [(512, 8, 0), (520, 13, 1)])
def test_which_prompts_run_on_pairs(device, dtype, d, n_head, pairs):
    """The persistent launch from 520 columns on, the others from 512 and 129 tokens."""
    cfg = small_cfg(n_layer=1, n_head=n_head, n_embd=d, n_ctx=140, vocab_size=101, dtype=dtype)
    gpt = load(cfg, make_model(cfg, 8))
    assert gpt.pairs() == -1
    for T, route, on in ((1, 1, pairs), (128, 1, pairs), (129, 0, 1), (64, 1, pairs)):
        gpt.prefill(synth.tokens(T, "prompt", T, cfg["vocab_size"]))
        assert (gpt.routes()[0], gpt.pairs()) == (route, on), T
    gpt.unloadBuffers()
