"""What a user of this framework has it do, as cases that can be timed.

The framework trains BLOOM-shaped models: decoder blocks written as word
scripts, run by the word machine on HIP kernels, and a driver for the whole
model with its AdamW step.  Four kinds of work make that up:

  block    one decoder block through its word script (host.Env): a training
           step (forward and backward) or the forward pass alone, by one of the
           three word sets the package ships -- `flash` (fused attention, head
           size 128), `mixed` (operator chain over 16-bit operand buffers, any
           head size) and `plain` (the operator stream of BlackRiver's own model
           scripts over the fp32 arena)
  model    BloomModel.step: embedding, blocks, final LayerNorm, tied LM head and
           loss, forward and backward
  adamw    BloomModel.optimizer_step: every parameter of a model
  logits   op.last_logits: the LM head on the last real token of every sequence
"""
import math

import numpy as np
import torch

from blackriver_amd import hip, host

GRADS = ["input_layernorm.weight_g", "input_layernorm.bias_g", "post_attention_layernorm.weight_g",
         "post_attention_layernorm.bias_g", "query_key_value.weight_g", "query_key_value.bias_g", "dense.weight_g",
         "dense.bias_g", "dense_h_to_4h.weight_g", "dense_h_to_4h.bias_g", "dense_4h_to_h.weight_g",
         "dense_4h_to_h.bias_g"]
MATRICES = ["query_key_value.weight", "dense.weight", "dense_h_to_4h.weight", "dense_4h_to_h.weight"]
VECTORS = ["input_layernorm.weight", "input_layernorm.bias", "post_attention_layernorm.weight",
           "post_attention_layernorm.bias", "query_key_value.bias", "dense.bias", "dense_h_to_4h.bias",
           "dense_4h_to_h.bias"]
MODEL_VECTORS = ["word_embeddings_layernorm.weight", "word_embeddings_layernorm.bias", "ln_f.weight", "ln_f.bias"]


def block(name, words, mode, hidden, head, batch, tokens, weights="f16", products="f16", padded=False):
    return {"name": name, "kind": "block", "words": words, "pass": mode, "hidden": hidden, "head": head, "batch": batch,
            "tokens": tokens, "weights": weights, "products": products, "padded": padded}


def listed():
    return [
        # the smallest step the tests and the smoke run take: launches and host work
        block("tiny-step", "flash", "step", 256, 128, 2, 32, padded=True),
        # fine-tuning on one short text: 78 tokens, a multiple of no tile
        block("short-step", "flash", "step", 1024, 128, 1, 78),
        # the benchmark's block: hidden 4096, 4 x 512 tokens
        block("headline-step", "flash", "step", 4096, 128, 4, 512),
        # a padded batch of ragged length, bf16 weights
        block("ragged-bf16-step", "flash", "step", 2048, 128, 3, 334, "bf16", "bf16", padded=True),
        # reading a long prompt: forward only
        block("long-forward", "flash", "forward", 4096, 128, 1, 2048),
        # head size 64: the operator chain, ragged length
        block("chain-step", "mixed", "step", 1024, 64, 4, 250),
        # BlackRiver's own operator stream with fp16 weights
        block("script-step", "plain", "step", 2048, 128, 2, 512, padded=True),
        # ... and as its scripts come: fp32 weights, fp32 products
        block("script-fp32-step", "plain", "step", 1024, 128, 2, 256, "float", "f32"),
        # three blocks of the benchmark's model with its 250880-word tied head, one 512-token sequence
        {"name": "model-step", "kind": "model", "layers": 3, "hidden": 4096, "head": 128, "vocab": 250880, "batch": 1,
         "tokens": 512, "weights": "f16", "products": "f16"},
        # a small model with an odd vocabulary: many short launches
        {"name": "small-model-step", "kind": "model", "layers": 2, "hidden": 512, "head": 128, "vocab": 32001,
         "batch": 2, "tokens": 100, "weights": "f16", "products": "f16"},
        # the optimizer after it: fp16 matrices with fp32 masters, many small vectors
        {"name": "adamw-step", "kind": "adamw", "layers": 2, "hidden": 2048, "head": 128, "vocab": 32000, "batch": 1,
         "tokens": 64, "weights": "f16", "products": "f16"},
        # next-word scores for eight sequences
        {"name": "last-logits", "kind": "logits", "hidden": 4096, "vocab": 250880, "batch": 8, "tokens": 128,
         "weights": "f16", "products": "f16"},
    ]


def log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def arena_tokens(tokens, heads):
    """Kernels between the fp32 arena and 16-bit products take the arena's tensors
    16-byte aligned: the ALiBi table [heads, tokens] and the mask [batch, tokens,
    tokens] in front of them have to fill whole quads of floats.  (The flash
    forward pass and fp32 products run at any length.)"""
    step = 2 if heads % 2 == 0 else 4
    return tokens // step * step


def draw(rng):
    """One more case of the same ranges: hidden sizes 256 .. 4096, 16 .. 2048
    tokens a step, every word set, storage type and head size."""
    kind = rng.choice(["block"] * 8 + ["model"] * 2 + ["adamw", "logits"])
    types = rng.choice([("f16", "f16"), ("f16", "f16"), ("bf16", "bf16")])
    if kind == "block":
        words = rng.choice(["flash", "flash", "mixed", "plain"])
        if words == "plain":
            types = rng.choice([("f16", "f16"), ("float", "f16"), ("float", "f32"), ("bf16", "bf16")])
        head = 128 if words == "flash" else rng.choice([64, 96, 128])
        most = 2048 if types[1] == "f32" else 4096
        hidden = head * log_uniform(rng, 256 // head, most // head)
        batch = rng.randint(1, 4)
        # a block keeps its LayerNorm statistics in vectors of `hidden` entries: no more tokens than that
        rows = min(hidden, 1024 if types[1] == "f32" or words != "flash" else 2048)
        tokens = log_uniform(rng, 16, rows // batch)
        mode = rng.choice(["step", "step", "forward"])
        if types[1] != "f32" and (words != "flash" or mode == "step"):
            tokens = arena_tokens(tokens, hidden // head)
        c = block("", words, mode, hidden, head, batch, tokens, *types,
                  padded=rng.random() < 0.5)
        del c["name"]
        return c
    if kind == "logits":
        return {"kind": "logits", "hidden": 64 * rng.randint(8, 64), "vocab": log_uniform(rng, 5000, 250880),
                "batch": rng.randint(1, 32), "tokens": rng.randint(16, 128), "weights": types[0], "products": types[1]}
    hidden = 128 * log_uniform(rng, 2, 24)
    batch = rng.randint(1, 3)
    tokens = arena_tokens(log_uniform(rng, 24, min(hidden, 1024) // batch), hidden // 128)
    return {"kind": kind, "layers": rng.randint(1, 3), "hidden": hidden, "head": 128,
            "vocab": log_uniform(rng, 1000, 60000), "batch": batch, "tokens": tokens, "weights": types[0],
            "products": types[1]}


# ------------------------------------------------------------------ plumbing
class _Memory:
    """A tensor of an environment as torch sees device memory; keeps its owner alive."""

    def __init__(self, owner, pointer, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (pointer, False), "version": 2}


def view(env, name):
    """The tensor `name` of the current hash as a torch tensor over the same memory."""
    code, on_device, shape, pointer = env.info(name)
    assert on_device, name
    t = torch.as_tensor(_Memory(env, pointer, shape, {hip.F32: "<f4", hip.F16: "<f2", hip.BF16: "<i2"}[code]),
                        device="cuda")
    return t.view(torch.bfloat16) if code == hip.BF16 else t


def boot():
    if not host.booted():
        torch.cuda.init()
        host.boot(0, 1 << 30)
        host.set_echo_loss(False)


def lengths(g, batch, tokens):
    """Real tokens of each right-padded sequence: between half and all of them."""
    return [int(n) for n in g.integers(max(2, tokens // 2), tokens + 1, batch)]


def mask_of(g, batch, tokens, padded):
    mask = np.ones((batch, tokens), np.int32)
    if padded:
        for b, n in enumerate(lengths(g, batch, tokens)):
            mask[b, n:] = 0
    return mask


def ids_of(g, batch, tokens, vocab):
    """Word ids with the frequencies text has: about 1 / rank."""
    return np.minimum(vocab ** g.random((batch, tokens)), vocab - 1).astype(np.int32)


def normal(t, gen, std, mean=0.0):
    t.normal_(mean, std, generator=gen)


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    boot()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    state = {"block": prepare_block, "model": prepare_model, "adamw": prepare_adamw,
             "logits": prepare_logits}[case["kind"]](case, seed, gen, np.random.default_rng(seed))
    torch.cuda.synchronize()
    return state


def prepare_block(case, seed, gen, rng):
    h, b, t = case["hidden"], case["batch"], case["tokens"]
    env = host.Env(1)
    env.execute(host.words_text("bloom.words"))
    env.execute("%d %d 1024 1e-05 model_dims" % (h, h // case["head"]))
    env.set("$DEVICE", "cuda")
    env.set("$WDTYPE", case["weights"])
    env.execute("'%s' op.gemm_precision create_layer_weight create_layer_grad zero_layer_grad" % case["products"])
    env.execute("%d %d dynamic_floats" % (b, t))
    env.execute("%d create_var %d %d create_dynamic" % (int(env.pop_number()) + 1024, b, t))
    env.execute("%d %d %d 3 'cuda' 'float' op.create 'dy' !" % (b, t, h))
    if case["words"] != "plain":
        env.execute("create_operand_buffers")
    env.execute("op.sync")
    for name in MATRICES:
        normal(view(env, name), gen, 0.02)
    for name in VECTORS:
        normal(view(env, name), gen, 0.02, 1.0 if name.endswith("layernorm.weight") else 0.0)
    normal(view(env, "xinput"), gen, 1.0)
    normal(view(env, "dy"), gen, 1.0)
    torch.cuda.synchronize()
    env.write("mask_", mask_of(rng, b, t, case["padded"]))
    env.execute("'yout_g' @ 'dy' @ op.copy")
    if case["words"] == "flash":
        env.execute("create_flash_buffers prepare_batch_flash op.sync")
    else:
        env.execute("prepare_batch op.sync")
    suffix = {"plain": "", "mixed": "_mixed", "flash": "_flash"}[case["words"]]
    if case["pass"] == "forward":
        text, outputs = "layer_forward" + suffix, ["xa"]
    else:
        # the operator-chain words add to yout_g in place, so a step of theirs starts from a copy of dy
        text = ("" if suffix == "_flash" else "'yout_g' @ 'dy' @ op.copy ") + "block_step" + suffix
        outputs = ["xa"] + GRADS
    return {"env": env, "program": env.build(text), "out": [view(env, n) for n in outputs]}


def new_model(case):
    return host.BloomModel(case["layers"], case["batch"], case["tokens"], case["hidden"], case["hidden"] // case["head"],
                           case["vocab"], 1e-5, case["weights"], case["products"])


def prepare_model(case, seed, gen, rng):
    model = new_model(case)
    model.init(seed, 0.02)
    out = [view(model.env, n) for n in ["word_embeddings.weight_g"] + [v + "_g" for v in MODEL_VECTORS]]
    for layer in range(1, case["layers"] + 1):
        model.env.change_hash(layer)
        out += [view(model.env, n) for n in GRADS]
    model.env.change_hash(0)
    return {"model": model, "ids": ids_of(rng, case["batch"], case["tokens"], case["vocab"]),
            "mask": mask_of(rng, case["batch"], case["tokens"], True), "out": out}


def prepare_adamw(case, seed, gen, rng):
    model = new_model(case)
    model.init(seed, 0.02)
    model.create_optimizer(lr=1e-3, weight_decay=0.01)
    out = []

    def parameter(name, matrix):
        normal(view(model.env, name + "_g"), gen, 1e-3)
        for suffix in ("", "_w32", "_m", "_v") if matrix else ("",):
            out.append(view(model.env, name + suffix))
    parameter("word_embeddings.weight", True)
    for name in MODEL_VECTORS:
        parameter(name, False)
    for layer in range(1, case["layers"] + 1):
        model.env.change_hash(layer)
        for name in MATRICES:
            parameter(name, layer <= 2)
        for name in VECTORS:
            parameter(name, False)
    model.env.change_hash(0)
    return {"model": model, "out": out}


def prepare_logits(case, seed, gen, rng):
    h, v, b, t = case["hidden"], case["vocab"], case["batch"], case["tokens"]
    env = host.Env(1)
    env.execute("'%s' op.gemm_precision" % case["products"])
    env.execute("%d %d 2 'cuda' '%s' op.create 'lm_head.weight' !" % (v, h, case["weights"]))
    env.execute("%d %d %d 3 'cuda' 'float' op.create 'x' !" % (b, t, h))
    env.execute("%d %d 2 'cuda' 'float' op.create 'logits' !" % (b, v))
    env.execute("8192 1 'cpu' 'int' op.create 'mask_buffer' !  'mask_buffer' @ 0 %d %d 2 op.view 'mask_' !" % (b, t))
    normal(view(env, "lm_head.weight"), gen, 0.02)
    normal(view(env, "x"), gen, 1.0)
    torch.cuda.synchronize()
    env.write("mask_", mask_of(rng, b, t, True))
    return {"env": env, "program": env.build("'x' @ 'mask_' @ 'lm_head.weight' @ 'logits' @ op.last_logits"),
            "out": [view(env, "logits")]}


# ------------------------------------------------------------------ run
def run(state):
    model = state.get("model")
    if model is None:
        state["env"].run(state["program"])
        return state["out"]
    if "ids" in state:
        return [model.step(state["ids"], state["mask"])] + state["out"]
    model.optimizer_step()
    return state["out"]


# ------------------------------------------------------------------ work
def work(case):
    h, b, t = case["hidden"], case["batch"], case["tokens"]
    n = b * t
    wb = 4 if case["weights"] == "float" else 2
    block_flops = 24.0 * n * h * h + 2.0 * n * (t + 1) * h      # four linear layers, the causal half of attention
    block_params, block_vectors = 12 * h * h, 13 * h
    if case["kind"] == "block":
        forward = block_params * wb + block_vectors * 4 + 2 * n * h * 4
        if case["pass"] == "forward":
            return {"bytes": forward, "flops": block_flops}
        return {"bytes": forward + n * h * 4 + (block_params + block_vectors) * 4, "flops": 3 * block_flops}
    v = case["vocab"]
    if case["kind"] == "logits":
        return {"bytes": v * h * wb + b * h * 4 + b * v * 4, "flops": 2.0 * b * v * h}
    matrices = case["layers"] * block_params + v * h
    vectors = case["layers"] * block_vectors + 4 * h
    if case["kind"] == "adamw":
        return {"bytes": matrices * 30 + vectors * 28, "flops": 15.0 * (matrices + vectors)}
    return {"bytes": matrices * (wb + 4) + vectors * 8, "flops": 3 * (case["layers"] * block_flops + 2.0 * n * h * v)}


def tolerance(case):
    """Four times what was seen: blocks against the same block in 64-bit torch
    (2-norm 9e-4 with fp16 products, 5.4e-3 with bf16, 5.8e-6 with fp32; largest
    entry 7.8e-3, 5.4e-2, 8.3e-5 of its scale), whole models on fused attention
    against the operator chain (largest entry, in the tied table's gradient, 0.09
    with fp16 and 0.13 with bf16)."""
    if case["kind"] == "adamw":
        # 32-bit element-wise arithmetic; a 16-bit weight may round to its neighbour
        return {"rel": 1e-4, "max": 1e-2}
    if case["kind"] == "logits":
        # 16-bit operands, one product summed in 32 bits
        return {"rel": 1e-5, "max": 1e-3}
    if case["products"] == "f32":
        return {"rel": 2.4e-5, "max": 3.5e-4}
    if case["products"] == "bf16":
        return {"rel": 2.2e-2, "max": 0.5 if case["kind"] == "model" else 0.22}
    return {"rel": 4e-3, "max": 0.35 if case["kind"] == "model" else 0.032}
