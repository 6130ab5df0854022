"""A layer of a few tokens in two launches (-m gpu) against the oracle's products of q8_1 activations: every format on either side, experts that
several tokens share, choices that are no expert, the smallest and largest sizes that it takes, replayed graphs."""

import numpy as np
import pytest
import torch

from helpers import QTYPES, assert_matches_f32_reference, random_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import synth
    import torch_ggml_ops
    from torch_ggml_ops import _native

    assert torch.cuda.is_available()
    return torch_ggml_ops, _native.lib, synth


def _bits(values):
    return values.to(torch.bfloat16).view(torch.int16).numpy().view(np.uint16)


def _expected(oracle, hidden, chosen, weights, gate, up, down, gate_up_type, down_type, n):
    """q8_1 products per slot; gate, up and their product rounded to bf16, the weighted sum in float64."""
    tokens, k = hidden.shape
    out = np.zeros((tokens, k))
    for t in range(tokens):
        for j, expert in enumerate(chosen[t].tolist()):
            if not 0 <= expert < gate.shape[0]:
                continue
            x = _bits(hidden[t : t + 1].cpu())
            g, u = (
                torch.from_numpy(oracle.mmq_forward(gate_up_type, x, w[expert].numpy(), n, k)).to(torch.bfloat16).float() for w in (gate, up)
            )
            activated = _bits(torch.nn.functional.silu(g) * u)
            out[t] += weights[t, j].item() * oracle.mmq_forward(down_type, activated, down[expert].numpy(), k, n)[0].astype(np.float64)
    return out.astype(np.float32)


def _layer(synth, tokens, top_k, experts, k, n, gate_up, down, seed):
    generator = torch.Generator().manual_seed(seed)
    chosen = torch.rand(tokens, experts, generator=generator).topk(top_k).indices
    weights = torch.rand(tokens, top_k, generator=generator) + 0.1
    gate, up = (synth.random_packed_weight(QTYPES[gate_up], (experts, n), k, seed=seed + s) for s in (1, 2))
    return random_bf16((tokens, k), seed=seed, scale=0.1), chosen, weights, gate, up, synth.random_packed_weight(QTYPES[down], (experts, k), n, seed=seed + 3)


def _check(tgo, lib, oracle, hidden, chosen, weights, gate, up, down, gate_up, down_type, n):
    types = QTYPES[gate_up], QTYPES[down_type]
    tokens, top_k = chosen.shape
    assert lib.tgo_moe_decode_workspace_bytes(tokens, top_k, gate.shape[0], hidden.shape[1], n, *types) > 0
    device = [t.cuda() for t in (chosen, weights, gate, up, down)]
    with torch.no_grad():
        actual = tgo.moe_layer(hidden, *device, *types, n)
        again = tgo.moe_layer(hidden, *device, *types, n)
    assert torch.equal(actual, again)
    # (fp32 sums in another order may round one of an expert's activations to the neighbouring bf16, which moves the scale of its block of 32
    # by 2^-8 at most: a sixteenth of the sum or less, so a few 1e-4 of the largest result)
    expected = _expected(oracle, hidden, chosen, weights, gate, up, down, *types, n)
    assert_matches_f32_reference(actual, expected, accumulate_noise=1e-3)
    return device


@pytest.mark.parametrize("gate_up,down", [("Q3_K", "Q4_K"), ("Q4_K", "Q5_K"), ("Q5_K", "Q6_K"), ("Q6_K", "IQ2_S"), ("IQ2_S", "Q3_K")])
@pytest.mark.parametrize(
    "tokens,top_k,experts,k,n",
    [(1, 8, 9, 2048, 512), (5, 3, 4, 1024, 512), (2, 1, 3, 2304, 256), (3, 6, 7, 4096, 1024), (6, 8, 8, 768, 768), (7, 5, 6, 2048, 256)],
)
def test_layer(ops, oracle, gate_up, down, tokens, top_k, experts, k, n):
    tgo, lib, synth = ops
    layer = _layer(synth, tokens, top_k, experts, k, n, gate_up, down, seed=tokens + k)
    _check(tgo, lib, oracle, *layer, gate_up, down, n)


def test_choices_that_are_no_expert_contribute_nothing(ops, oracle):
    """Also where a whole token has none, where a token names one expert twice, and with a workspace of NaN, of which the slots without an expert are
    never written."""
    from torch_ggml_ops import _native

    tgo, lib, synth = ops
    hidden, chosen, weights, *experts = _layer(synth, 5, 3, 5, 1024, 512, "Q6_K", "Q4_K", seed=11)
    chosen[1] = torch.tensor([-1, 5, 1 << 40])
    chosen[2, 1] = -7
    chosen[3] = torch.tensor([4, 2, 4])
    device = _check(tgo, lib, oracle, hidden, chosen, weights, *experts, "Q6_K", "Q4_K", 512)
    with torch.no_grad():
        expected = tgo.moe_layer(hidden, *device, QTYPES["Q6_K"], QTYPES["Q4_K"], 512)
    sizes = (5, 3, 5, 1024, 512, QTYPES["Q6_K"], QTYPES["Q4_K"])
    workspace = torch.full((lib.tgo_moe_decode_workspace_bytes(*sizes),), 0xFF, dtype=torch.uint8, device="cuda")
    assert workspace.view(torch.bfloat16).isnan().all()
    actual = torch.empty_like(expected)
    pointers = [t.data_ptr() for t in (hidden, *device, actual, workspace)]
    _native.check(lib.tgo_moe_decode(*pointers, *sizes, _native.stream_of(hidden.device)))
    assert torch.equal(actual, expected) and not actual[1].any()
    assert workspace.view(torch.bfloat16).view(15, 512)[[3, 4, 5, 7]].isnan().all()


def test_graph(ops):
    """Replays with other choices and activations in the captured tensors, with eager calls in between."""
    tgo, lib, synth = ops
    hidden, chosen, weights, *experts = _layer(synth, 4, 4, 16, 1024, 512, "IQ2_S", "Q6_K", seed=21)
    chosen, weights, *experts = (t.cuda() for t in (chosen, weights, *experts))
    arguments = (hidden, chosen, weights, *experts, QTYPES["IQ2_S"], QTYPES["Q6_K"], 512)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.no_grad(), torch.cuda.stream(stream):
        tgo.moe_layer(*arguments)
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph, stream=stream):
        captured = tgo.moe_layer(*arguments)
    for replay in range(4):
        hidden.copy_(random_bf16(hidden.shape, seed=50 + replay, scale=0.1))
        chosen.copy_(torch.rand(4, 16, generator=torch.Generator().manual_seed(replay)).topk(4).indices)
        graph.replay()
        with torch.no_grad():
            assert torch.equal(captured, tgo.moe_layer(*arguments))
