"""The work that programs have this library do, as cases that can be timed: decode, prefill and training through the
public operators, dense and mixture-of-experts, over the sizes and weight formats in use.

A case is a dict of plain values.  Its "kind" says which calls a pass makes:

  dense    ``mmq`` without a gradient: one projection of a decode step or of a prefill, or the logits of a sampler
  train    ``mmq`` and the gradient of its input: a frozen packed projection below trained adapters
  qkv      ``mmq_multi`` of three projections and the gradient of their input: grouped-query attention in training
  pair     ``grouped_mmq_pair`` and the gradient of its input on expert-sorted rows: gate and up of a trained layer
  moe      ``moe_layer`` without a gradient, called from Python: a decode step, a chunk or a prefill
  graph    eight ``moe_layer`` calls with weights of their own in one HIP graph, replayed: a serving loop's decode step
  moe_train  ``moe_layer`` with the gradients of its input and of the routing weights
  head     ``chunked_lm_head_loss`` and its gradient: the loss of a training step

Everything is synthetic: packed blocks of random bytes with scales that give weights of the size a trained model has,
normally distributed activations, and top-k routing with a skew over the experts.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "torch-ggml-ops_amd"))
import torch_ggml_ops as tgo  # noqa: E402

TYPES = {"Q3_K": 11, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14, "IQ2_S": 22}
BLOCK_BYTES = {"Q3_K": 110, "Q4_K": 144, "Q5_K": 176, "Q6_K": 210, "IQ2_S": 82}
# (byte offset of a block's fp16 scale, its middle value): weights of about 0.02 with the formats' own integers; the
# second field of Q4_K and Q5_K is the scale of the minimum, which centres the weights
SCALES = {
    "Q3_K": ((108, 5e-4),), "Q4_K": ((0, 1e-4), (2, 7.5e-4)), "Q5_K": ((0, 6.5e-5), (2, 1e-3)),
    "Q6_K": ((208, 1.2e-5),), "IQ2_S": ((0, 4e-4),),
}
GRAPH_LAYERS = 8
HEAD = (248320, 2048)   # vocabulary x features of the model family whose shapes the operators are used with


def listed():
    return [
        # the query projection of one decoded token: the smallest call, whose time is its launch
        {"name": "proj_decode_1", "kind": "dense", "type": "Q3_K", "rows": 1, "n": 4096, "k": 2048},
        # a feed-forward projection of a large dense model for a few sequences: bound by the packed bytes
        {"name": "ffn_decode_5", "kind": "dense", "type": "Q4_K", "rows": 5, "n": 28672, "k": 8192},
        # a short ragged prompt, and an output width that is no multiple of a tile
        {"name": "proj_prefill_517", "kind": "dense", "type": "Q6_K", "rows": 517, "n": 5003, "k": 4096},
        # an attention projection in training
        {"name": "proj_train_4096", "kind": "train", "type": "Q5_K", "rows": 4096, "n": 4096, "k": 2048},
        # query, key and value of a layer with four query heads to each key head, in training
        {"name": "qkv_train_2048", "kind": "qkv", "type": "Q4_K", "rows": 2048, "n": 4096, "k": 4096},
        # a mixture-of-experts layer of one decoded token, called from Python
        {"name": "moe_decode_1", "kind": "moe", "type": "IQ2_S", "down": "Q6_K", "tokens": 1, "experts": 256, "top_k": 8,
         "k": 2048, "n": 512, "skew": 0.3},
        # the layers of a decode step for a few sequences as a serving loop replays them
        {"name": "moe_decode_6_graph", "kind": "graph", "type": "IQ2_S", "down": "Q6_K", "tokens": 6, "experts": 256, "top_k": 8,
         "k": 2048, "n": 512, "skew": 0.3},
        # a prefill chunk mixed into decoding: a few rows for every expert
        {"name": "moe_chunk_97", "kind": "moe", "type": "Q3_K", "down": "Q4_K", "tokens": 97, "experts": 256, "top_k": 8,
         "k": 2048, "n": 512, "skew": 0.3},
        # a prompt
        {"name": "moe_prefill_2048", "kind": "moe", "type": "IQ2_S", "down": "Q4_K", "tokens": 2048, "experts": 256, "top_k": 8,
         "k": 2048, "n": 512, "skew": 0.3},
        # a whole layer in training
        {"name": "moe_train_4096", "kind": "moe_train", "type": "IQ2_S", "down": "Q5_K", "tokens": 4096, "experts": 256, "top_k": 8,
         "k": 2048, "n": 512, "skew": 0.3},
        # the benchmark's workload: gate and up with Zipf-skewed routing, forward and backward
        {"name": "pair_train_8192", "kind": "pair", "type": "Q5_K", "tokens": 8192, "experts": 256, "top_k": 8, "k": 2048, "n": 512,
         "skew": 1.1},
        # the loss of a training step, with a last chunk that is not full
        {"name": "head_loss_1000", "kind": "head", "type": "Q6_K", "rows": 1000, "n": HEAD[0], "k": HEAD[1]},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _experts(rng, low, high):
    """A mixture-of-experts geometry and a token count whose largest product stays at that of the listed pair."""
    experts, top_k = rng.choice([(256, 8), (128, 8), (64, 6)])
    k, n = rng.choice([(2048, 512), (2048, 768), (1024, 512), (4096, 1024)])
    most = 8192 * 8 * 2048 * 512 // (top_k * k * n)
    return {"tokens": _log(rng, low, min(high, most)), "experts": experts, "top_k": top_k, "k": k, "n": n, "skew": rng.choice([0.3, 0.7, 1.1])}


def draw(rng):
    kind = rng.choice(["dense", "dense", "train", "qkv", "pair", "moe", "moe", "graph", "moe_train", "head"])
    quant = rng.choice(sorted(TYPES))
    if kind in ("dense", "train", "qkv"):
        k = 256 * _log(rng, 2, 32)
        n = _log(rng, 512, 28672)
        if kind == "dense" and rng.random() < 0.5:
            rows = _log(rng, 1, 64)
        else:
            rows = _log(rng, 64, max(65, min(16384, 2**38 // (n * k))))
        if kind == "qkv":
            n = max(512, n // 4 * 4)
        elif rng.random() < 0.5:
            n = (n + 127) // 128 * 128   # widths are multiples of a head's width more often than not
        return {"kind": kind, "type": quant, "rows": rows, "n": n, "k": k}
    if kind == "head":
        return {"kind": kind, "type": rng.choice(["Q4_K", "Q5_K", "Q6_K"]), "rows": _log(rng, 64, 1000), "n": _log(rng, 32000, HEAD[0]),
                "k": HEAD[1]}
    if kind == "pair":
        return {"kind": kind, "type": quant, **_experts(rng, 256, 8192)}
    down = rng.choice(["Q4_K", "Q5_K", "Q6_K"])
    if kind == "graph":
        case = {"kind": kind, "type": quant, "down": down, **_experts(rng, 1, 16)}
    elif kind == "moe":
        case = {"kind": kind, "type": quant, "down": down, **(_experts(rng, 1, 64) if rng.random() < 0.5 else _experts(rng, 64, 4096))}
    else:
        case = {"kind": kind, "type": quant, "down": down, **_experts(rng, 256, 4096)}
    return case


def _weight(quant, leading, k, generator):
    blocks = math.prod(leading) * (k // 256)
    data = torch.randint(0, 256, (blocks, BLOCK_BYTES[quant]), dtype=torch.uint8, device="cuda", generator=generator)
    for offset, middle in SCALES[quant]:
        scale = (torch.rand(blocks, device="cuda", generator=generator) * 0.5 + 0.75) * middle
        data[:, offset : offset + 2] = scale.to(torch.float16).view(torch.uint8).reshape(-1, 2)
    return data.reshape(*leading, (k // 256) * BLOCK_BYTES[quant])


def _normal(shape, generator, scale=1.0):
    return (torch.randn(*shape, device="cuda", generator=generator) * scale).to(torch.bfloat16)


def _choices(case, generator):
    """(slot_experts, slot_weights) of a router: normal logits plus a power law over the experts in random order."""
    tokens, experts, top_k = case["tokens"], case["experts"], case["top_k"]
    logits = torch.randn(tokens, experts, device="cuda", generator=generator)
    law = -case["skew"] * torch.arange(1, experts + 1, device="cuda", dtype=torch.float32).log()
    logits += law[torch.randperm(experts, device="cuda", generator=generator)]
    weights, chosen = torch.softmax(logits, dim=-1).topk(top_k, dim=-1)
    return chosen.contiguous(), (weights / weights.sum(dim=-1, keepdim=True)).contiguous()


def _layer(case, generator):
    experts, k, n = case["experts"], case["k"], case["n"]
    chosen, weights = _choices(case, generator)
    return {
        "hidden": _normal((case["tokens"], k), generator), "chosen": chosen, "weights": weights,
        "gate": _weight(case["type"], (experts, n), k, generator), "up": _weight(case["type"], (experts, n), k, generator),
        "down": _weight(case["down"], (experts, k), n, generator),
    }


def _call(case, layer):
    return tgo.moe_layer(
        layer["hidden"], layer["chosen"], layer["weights"], layer["gate"], layer["up"], layer["down"],
        TYPES[case["type"]], TYPES[case["down"]], case["n"],
    )


def _widths(case):
    return (case["n"], case["n"] // 4, case["n"] // 4) if case["kind"] == "qkv" else (case["n"],)


def prepare(case, seed):
    generator = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    state = {"case": case}
    if kind in ("dense", "train", "qkv", "head"):
        rows, k = case["rows"], case["k"]
        state["x"] = _normal((rows, k), generator).requires_grad_(kind != "dense")
        state["w"] = [_weight(case["type"], (n,), k, generator) for n in _widths(case)]
        if kind == "head":
            targets = torch.randint(0, case["n"], (rows,), device="cuda", generator=generator)
            # (a prompt's tokens are not counted)
            state["targets"] = torch.where(torch.rand(rows, device="cuda", generator=generator) < 0.1, -100, targets)
        elif kind != "dense":
            state["grads"] = [_normal((rows, n), generator, 1e-2) for n in _widths(case)]
    elif kind == "pair":
        chosen, _ = _choices(case, generator)
        row_index, _, experts, offsets = tgo.route(chosen, case["experts"])
        rows = row_index.numel()
        state["x"] = _normal((case["tokens"], case["k"]), generator).index_select(0, row_index).requires_grad_()
        state["w"] = [_weight(case["type"], (case["experts"], case["n"]), case["k"], generator) for _ in range(2)]
        state["groups"] = (experts, offsets)
        state["grads"] = [_normal((rows, case["n"]), generator, 1e-2) for _ in range(2)]
    elif kind == "graph":
        state["layers"] = [_layer(case, generator) for _ in range(GRAPH_LAYERS)]
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.no_grad():
            with torch.cuda.stream(stream):
                _call(case, state["layers"][0])
            torch.cuda.current_stream().wait_stream(stream)
            torch.cuda.synchronize()
            state["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(state["graph"], stream=stream):
                state["out"] = [_call(case, layer) for layer in state["layers"]]
    else:
        state["layer"] = _layer(case, generator)
        if kind == "moe_train":
            state["layer"]["hidden"].requires_grad_()
            state["layer"]["weights"].requires_grad_()
            state["grad"] = _normal((case["tokens"], case["k"]), generator, 1e-2)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "graph":
        state["graph"].replay()
        return state["out"]
    if kind == "moe":
        with torch.no_grad():
            return _call(case, state["layer"])
    if kind == "moe_train":
        layer = state["layer"]
        out = _call(case, layer)
        return (out, *torch.autograd.grad(out, (layer["hidden"], layer["weights"]), state["grad"]))
    quant = TYPES[case["type"]]
    x = state["x"]
    if kind == "dense":
        with torch.no_grad():
            return tgo.mmq(x, state["w"][0], quant, case["n"])
    if kind == "head":
        loss = tgo.chunked_lm_head_loss(x, state["w"][0], state["targets"], quant, case["n"])
        return (loss, *torch.autograd.grad(loss, x))
    if kind == "train":
        outputs = (tgo.mmq(x, state["w"][0], quant, case["n"]),)
    elif kind == "qkv":
        outputs = tgo.mmq_multi(x, state["w"], [quant] * 3, _widths(case))
    else:
        outputs = tgo.grouped_mmq_pair(x, *state["w"], *state["groups"], quant, case["n"])
    return (*outputs, *torch.autograd.grad(outputs, x, state["grads"]))


def _packed(quant, rows, k):
    return rows * (k // 256) * BLOCK_BYTES[quant]


def work(case):
    """Packed weights, activations, cotangents and results once each in and out (bf16), and the products' operations.  A
    layer reads the experts that its tokens choose: those that even routing would reach."""
    kind, k, n = case["kind"], case["k"], case["n"]
    if kind in ("dense", "train", "qkv", "head"):
        rows, width = case["rows"], sum(_widths(case))
        flops = 2 * rows * width * k
        moved = _packed(case["type"], width, k) + 2 * rows * k
        if kind == "head":
            # (the logits need not leave the chip)
            return {"bytes": moved + 2 * rows * k, "flops": 2 * flops}
        moved += 2 * rows * width
        return {"bytes": moved, "flops": flops} if kind == "dense" else {"bytes": moved + 2 * rows * (width + k), "flops": 2 * flops}
    tokens, experts, top_k = case["tokens"], case["experts"], case["top_k"]
    slots = tokens * top_k
    active = experts * (1 - (1 - top_k / experts) ** tokens)
    pair = 2 * active * _packed(case["type"], n, k)
    if kind == "pair":
        return {"bytes": pair + 2 * slots * (2 * k + 4 * n), "flops": 8 * slots * n * k}
    moved = pair + active * _packed(case["down"], k, n) + 2 * tokens * 2 * k + 12 * slots
    flops = 6 * slots * n * k
    if kind == "graph":
        return {"bytes": GRAPH_LAYERS * moved, "flops": GRAPH_LAYERS * flops}
    if kind == "moe":
        return {"bytes": moved, "flops": flops}
    return {"bytes": moved + 2 * tokens * 2 * k + 4 * slots, "flops": 2 * flops}


def tolerance(case):
    """bf16 results of 8-bit activations.  Operands of one product may be rounded to fp16 or kept as integers; the steps
    of a layer round to bf16 and quantize again in between."""
    if case["kind"] in ("moe", "graph", "moe_train"):
        return {"rel": 1e-2, "max": 0.1}
    return {"rel": 5e-3, "max": 0.05}
