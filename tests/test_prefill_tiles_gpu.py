"""Long prompts against the CPU oracle: rows on both sides of the edges of the larger tiles, widths that are no multiple of 128 or of a step
of 32, both weight dtypes. Widths of 512 and more run on pairs (csrc/gemm_pair.hip), 456 in the tiles of csrc/gemm_split.hip, which
test_prefill_pairs_gpu.py holds the others to as well."""
import numpy as np
import pytest

from oracle import ref
from webgpt_amd import synth
from webgpt_amd.model import GPT

from helpers import close, make_model, oracle_weights, small_cfg, worst

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "int8"])
@pytest.mark.parametrize("d,n_head,rows", [(768, 12, (961, 960, 943, 865)), (744, 6, (513, 385, 289)), (1000, 10, (300, 193)), (456, 6, (1024, 700, 257)),
                                           (1600, 25, (300, 129))])
def test_prompts_against_oracle(device, dtype, d, n_head, rows):
    """Logits, cache rows and the residual rows of a layer's four products (the last one from all rows of both)."""
    cfg = small_cfg(n_layer=1, n_head=n_head, n_embd=d, n_ctx=1024, vocab_size=97, dtype=dtype)
    tensors = make_model(cfg, d)
    gpt = GPT(None, "char", tensors=tensors, params=synth.model_params(cfg))
    gpt.initialize()
    w, p = oracle_weights(tensors, cfg), synth.model_params(cfg)
    for T in rows:
        tokens = synth.tokens(T, "prompt", T, cfg["vocab_size"])
        want, taps, kv = ref.forward(p, w, tokens, want_taps=True, want_kv=True)
        got = gpt.prefill(tokens)
        assert close(got, want), (T, worst(got, want))
        for j, name in enumerate("kv"):
            rows_got = gpt.tap(f"kv0_{name}")
            assert close(rows_got, kv[0, j]), (T, name, worst(rows_got, kv[0, j]))
        # near zero a residual value's error is that of its terms: 1e-4 of the rows' root mean square, as for short prompts
        rows_got, exp = gpt.tap("residual", T), taps[ref.tap_names(1).index("block0_r2")]
        assert close(rows_got, exp, atol=1e-4 * float(np.sqrt(np.mean(exp ** 2)))), T
    gpt.unloadBuffers()
