"""The work that a user of this framework has it do, as cases that can be timed and compared.

A case is a dict of plain values. `kind` says which public entry points a pass goes through:

  prefill   GPT.run on a whole window: the prompt in, the logits of its last token out
  greedy    GPT.run on a prompt, then GPT.decode_greedy: tokens, and the logits of the last step
  generate  GPT.generate, the sampling loop of a chat or completion program (top_k, temperature)
  loop      GPT.run once per token with the logits on the host each time: a program with its own sampling
  blocks    a forward assembled from the instruction blocks (Embed, LayerNorm, Attention, FastMatMul, Gelu,
            Residual, DeEmbed), as a program with a model of its own builds it

with the model's dimensions beside it, the prompt length `T` and the number of tokens `n`. dtype "int8" is the
weight-only int8 form of the linear layers. Weights are drawn, not trained; the shapes are those of synth.CONFIGS or
generic ones.
"""
import math
import random

import numpy as np
import torch

from webgpt_amd import blocks, synth
from webgpt_amd.blocks import (AttentionBlock, DeEmbedBlock, EmbedBlock, FastMatMulBlock, GeluBlock, LayerNormBlock,
                               ResidualBlock, SoftmaxBlock)
from webgpt_amd.model import GPT

_DIMS = ("n_layer", "n_head", "n_embd", "n_ctx", "vocab_size")


def _case(kind, config, **more):
    c = {"kind": kind, "dtype": synth.CONFIGS[config]["dtype"]}
    c.update({k: synth.CONFIGS[config][k] for k in _DIMS})
    c.update(more)
    return c


def listed():
    generic = dict(n_layer=4, n_head=12, n_embd=576, n_ctx=512, vocab_size=5003, dtype="f32")
    return [
        # the character-level model, its program's defaults (80 tokens, top_k 2): the smallest launches there are
        _case("generate", "toy", name="toy-chat", T=64, n=80, top_k=2, temperature=1.0),
        # a model of no benchmarked shape (head size 48, odd vocabulary), odd prompt, short answer
        dict(generic, name="generic-greedy", kind="greedy", T=37, n=24),
        # the reference's own loop: GPT.run per token, logits to the host, from a short prompt
        _case("loop", "gpt2-117m", name="117m-loop", T=13, n=12),
        # the benchmark's prompt and a long ragged one: time to the first token
        _case("prefill", "gpt2-117m", name="117m-prefill-128", T=128),
        _case("prefill", "gpt2-117m", name="117m-prefill-943", T=943),
        # the headline decode: 128-token prompt, greedy continuation
        _case("greedy", "gpt2-117m", name="117m-greedy", T=128, n=128),
        # text completion with the usual sampling options
        _case("generate", "gpt2-117m", name="117m-sampled", T=45, n=48, top_k=40, temperature=0.9),
        _case("prefill", "gpt2-345m", name="345m-prefill-512", T=512),
        _case("greedy", "gpt2-774m", name="774m-greedy", T=64, n=48),
        # the weight-only int8 model: a prompt, and a continuation
        _case("prefill", "gpt2-1.5b-int8", name="1.5b-int8-prefill", T=300),
        _case("greedy", "gpt2-1.5b-int8", name="1.5b-int8-greedy", T=16, n=32),
        # a forward of two layers from the instruction blocks, whole window, as the reference's GPT.run chains them
        _case("blocks", "gpt2-117m", name="blocks-window", n_layer=2, T=100),
    ]


def _between(rng, lo, hi):
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    """One more case: any kind, the configured models and generic ones, prompts from one token to the whole context."""
    kind = rng.choice(["prefill", "prefill", "greedy", "generate", "loop", "blocks"])
    which = rng.choice(["toy", "gpt2-117m", "gpt2-117m", "gpt2-345m", "gpt2-774m", "gpt2-1.5b-int8", "generic", "generic", "generic"])
    if kind == "blocks" and which in ("gpt2-774m", "gpt2-1.5b-int8"):
        which = "gpt2-345m"
    if which == "generic":
        hs = rng.choice([16, 32, 40, 48, 64, 64, 80, 96, 128])
        c = dict(n_layer=rng.randint(2, 8), n_head=max(1, _between(rng, 64, 1280) // hs), n_embd=0,
                 n_ctx=rng.choice([128, 256, 512, 1000, 1024]), vocab_size=_between(rng, 65, 50257),
                 dtype=rng.choice(["f32", "f32", "int8"]) if kind != "blocks" else "f32", kind=kind)
        c["n_embd"] = c["n_head"] * hs
    else:
        c = _case(kind, which)
    if kind == "blocks":
        c["n_layer"] = rng.randint(1, 3)
    if kind == "prefill" or kind == "blocks":
        c["T"] = _between(rng, 1, c["n_ctx"])
        return c
    large = which in ("gpt2-774m", "gpt2-1.5b-int8")
    c["n"] = _between(rng, 4, 16 if kind == "loop" else 32 if large else 96)
    c["T"] = _between(rng, 1, c["n_ctx"] - c["n"])
    if kind == "generate":
        c["top_k"] = min(rng.choice([1, 2, 3, 5, 10, 40, 100]), c["vocab_size"])
        c["temperature"] = round(rng.uniform(0.6, 1.2), 3)
    return c


class _Values:
    """Normal values on the host, drawn once per state; a tensor is a run of them at a place of its own."""

    def __init__(self, seed, most):
        g = torch.Generator(device="cuda").manual_seed(int(seed))
        self.pool = torch.randn(most + 65536, generator=g, device="cuda").cpu().numpy()
        self.rng = np.random.default_rng(int(seed))

    def take(self, *shape):
        n = int(np.prod(shape))
        at = 16 * int(self.rng.integers(0, (self.pool.size - n) // 16 + 1))
        return self.pool[at:at + n].reshape(shape)


def _tensors(case, seed):
    """The weight directory of a drawn model: matrices and embeddings of std 0.02, LayerNorm gains around 1; the
    int8 form as quantising such matrices per column gives it."""
    d, V, ctx, int8 = case["n_embd"], case["vocab_size"], case["n_ctx"], case["dtype"] == "int8"
    most = max(V * d, ctx * d, 4 * d * d)
    v = _Values(seed, most)
    table = v.pool[:V * d].reshape(V, d).copy()
    small = (v.pool[:8 * d + 65536] * np.float32(0.1)).copy()
    if int8:
        words = np.clip(np.rint(v.pool[:4 * d * d + 65536] * np.float32(30.0)), -127, 127).astype(np.int8).view(np.int32)
    np.multiply(v.pool, np.float32(0.02), out=v.pool)
    np.multiply(table, np.float32(0.02), out=table)

    def few(n, centre=0.0, scale=1.0):
        at = int(v.rng.integers(0, small.size - n))
        return (small[at:at + n] * np.float32(scale) + np.float32(centre)).astype(np.float32)

    t = {"transformer.wte.weight": table, "transformer.wpe.weight": v.take(ctx, d),
         "transformer.ln_f.weight": few(d, 1.0), "transformer.ln_f.bias": few(d)}
    for i in range(case["n_layer"]):
        p = f"transformer.h.{i}."
        for ln in ("ln_1", "ln_2"):
            t[p + ln + ".weight"], t[p + ln + ".bias"] = few(d, 1.0), few(d)
        for stem, K, N in (("attn.c_attn", d, 3 * d), ("attn.c_proj", d, d), ("mlp.c_fc", d, 4 * d), ("mlp.c_proj", 4 * d, d)):
            t[p + stem + ".bias"] = few(N, 0.0, 0.2)
            if int8:
                n = K * (N // 4)
                at = int(v.rng.integers(0, words.size - n))
                t[p + stem + ".weight.q"] = words[at:at + n].reshape(K, N // 4)
                t[p + stem + ".weight.scale"] = few(N, 0.085, 0.05)
            else:
                t[p + stem + ".weight"] = v.take(K, N)
    return t


class _Model:
    """A loaded model and the prompt that a program holds; gives the device memory back with the state."""

    def __init__(self, case, seed):
        self.case, self.seed = case, int(seed)
        self.tokens = [int(i) for i in np.random.default_rng(int(seed) + 7).integers(0, case["vocab_size"], case["T"] + case.get("n", 0))]
        self.gpt = GPT(None, "bpe", tensors=_tensors(case, seed), params={k: case[k] for k in _DIMS})
        self.gpt.initialize()

    def __del__(self):
        if hasattr(self, "gpt"):
            self.gpt.unloadBuffers()


class _Blocks:
    """Weights of a model in device buffers, for a forward that the program chains itself."""

    def __init__(self, case, seed):
        self.case = case
        blocks.initializeOperations(blocks.Device(0))
        d, V = case["n_embd"], case["vocab_size"]
        self.buffers = {}
        for name, a in _tensors(case, seed).items():
            if name.endswith("c_attn.weight"):  # Q, K and V apart, as the reference's loader leaves them
                for j, part in enumerate("qkv"):
                    self.buffers[name + "." + part] = blocks.init_tensor(np.ascontiguousarray(a[:, j * d:(j + 1) * d]), [d, d])
            elif name.endswith("c_attn.bias"):
                for j, part in enumerate("qkv"):
                    self.buffers[name + "." + part] = blocks.init_tensor(a[j * d:(j + 1) * d], [d])
            else:
                self.buffers[name] = blocks.init_tensor(a, list(a.shape))
        self.tokens = np.random.default_rng(int(seed) + 7).integers(0, V, case["T"]).astype(np.int32)

    def __del__(self):
        for b in getattr(self, "buffers", {}).values():
            b.destroy()


def prepare(case, seed):
    return (_Blocks if case["kind"] == "blocks" else _Model)(case, seed)


def _run_blocks(s):
    c, b = s.case, s.buffers
    T, d, H, V = c["T"], c["n_embd"], c["n_head"], c["vocab_size"]
    passes, keep = [], []

    def add(inst):
        passes.extend(inst["passes"])
        keep.append(inst)
        return inst["resultBuffer"]

    x = add(EmbedBlock.newInstance(s.tokens, T, d, V, [b["transformer.wte.weight"]], b["transformer.wpe.weight"], ResidualBlock))
    for i in range(c["n_layer"]):
        p = f"transformer.h.{i}."
        h = add(LayerNormBlock.newInstance(T, d, x, b[p + "ln_1.weight"], b[p + "ln_1.bias"]))
        qkv = [b[p + "attn.c_attn." + kind + "." + part] for part in "qkv" for kind in ("weight", "bias")]
        h = add(AttentionBlock.newFusedInstance(T, d, 1 / math.sqrt(d // H), H, d // H, h, *qkv, b[p + "attn.c_proj.weight"],
                                                b[p + "attn.c_proj.bias"], FastMatMulBlock, SoftmaxBlock))
        x = add(ResidualBlock.newInstance(T, d, h, x))
        h = add(LayerNormBlock.newInstance(T, d, x, b[p + "ln_2.weight"], b[p + "ln_2.bias"]))
        h = add(FastMatMulBlock.newInstance(T, 4 * d, d, h, b[p + "mlp.c_fc.weight"], b[p + "mlp.c_fc.bias"]))
        h = add(GeluBlock.newInstance(T, 4 * d, h))
        h = add(FastMatMulBlock.newInstance(T, d, 4 * d, h, b[p + "mlp.c_proj.weight"], b[p + "mlp.c_proj.bias"]))
        x = add(ResidualBlock.newInstance(T, d, h, x))
    h = add(LayerNormBlock.newInstance(T, d, x, b["transformer.ln_f.weight"], b["transformer.ln_f.bias"]))
    logits = add(DeEmbedBlock.newInstance(d, V, V, T, V, h, [b["transformer.wte.weight"]]))
    blocks.run_passes(passes)
    out = {"logits": logits.download(), "residual": x.download().reshape(T, d)}
    blocks.clearOperationCache()
    return out


def run(s):
    c = s.case
    if c["kind"] == "blocks":
        return _run_blocks(s)
    gpt, prompt = s.gpt, s.tokens[:c["T"]]
    if c["kind"] == "prefill":
        return {"logits": gpt.run(prompt)}
    if c["kind"] == "greedy":
        first = gpt.run(prompt)
        ids, last = gpt.decode_greedy(int(np.argmax(first)), c["n"], want_logits=True)
        return {"first": first, "ids": ids, "last": last}
    if c["kind"] == "loop":
        return {"logits": np.stack([gpt.run(s.tokens[:c["T"] + i]) for i in range(c["n"] + 1)])}
    random.seed(s.seed)
    ids = np.array(list(gpt.generate(prompt, c["n"], c["top_k"], c["temperature"])), np.int32)
    return {"ids": ids, "next": gpt.run(prompt + [int(i) for i in ids])}


def work(case):
    """Each weight once per forward (the table's rows of the prompt, and the whole table for the logits), the keys and
    values of the context once per step, the activations of a prefill not at all; two operations per multiply-add."""
    L, d, V, T = case["n_layer"], case["n_embd"], case["vocab_size"], case["T"]
    linear = L * 12 * d * d * (1 if case["dtype"] == "int8" else 4) + 4 * L * 13 * d + (4 * L * 9 * d if case["dtype"] == "int8" else 0)
    table = 4 * V * d

    def window(T):
        return linear + table + 8 * T * d + 8 * L * d * T, 2 * T * 12 * L * d * d + 2 * L * T * (T + 1) * d + 2 * V * d

    def step(t):  # one token on top of t positions
        return linear + table + 8 * L * d * (t + 1), 24 * L * d * d + 4 * L * d * (t + 1) + 2 * V * d

    nbytes, flops = window(T)
    if case["kind"] in ("greedy", "loop"):
        steps = [step(T + i) for i in range(case["n"])]
    elif case["kind"] == "generate":  # the first token from the window, the others by steps; then the window that gives "next"
        steps = [step(T + i) for i in range(case["n"])]
    else:
        steps = []
    return {"bytes": nbytes + sum(s[0] for s in steps), "flops": flops + sum(s[1] for s in steps)}


def tolerance(case):
    """The same forward in 64 bits is 3e-7 (toy) to 1.8e-6 (48 layers, int8) away in norm and at most 8.3e-6 of the root
    mean square in one logit, whichever way the sums are ordered: four times that. Ids are compared as they are; `differ`
    leaves room for a tie at the end of a continuation."""
    return {"rel": 7e-6, "max": 3.5e-5, "differ": 0.01}
