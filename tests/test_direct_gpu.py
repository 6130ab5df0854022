"""Calls without a gradient that skip the dispatcher (-m gpu): the bits of the registered operators, and everything that is
not such a call still reaches those."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from helpers import QTYPES, random_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tgo():
    import torch_ggml_ops

    assert torch.cuda.is_available()
    return torch_ggml_ops


def _layer(tokens, top_k=4, experts=12, k=512, n=256):
    import synth

    generator = torch.Generator().manual_seed(tokens)
    chosen = torch.rand(tokens, experts, generator=generator).topk(top_k).indices.cuda()
    weights = torch.rand(tokens, top_k, generator=generator).cuda()
    gate, up = (synth.random_packed_weight(QTYPES["IQ2_S"], (experts, n), k, seed=s).cuda() for s in (1, 2))
    down = synth.random_packed_weight(QTYPES["Q4_K"], (experts, k), n, seed=3).cuda()
    return random_bf16((tokens, k), seed=4), chosen, weights, gate, up, down, QTYPES["IQ2_S"], QTYPES["Q4_K"], n


@pytest.mark.parametrize("tokens", (1, 40, 1500))
def test_layer_has_the_operators_bits(tgo, tokens):
    hidden, chosen, weights, gate, up, down, *rest = _layer(tokens)
    with_gradient = tgo.moe_layer(hidden.clone().requires_grad_(), chosen, weights, gate, up, down, *rest)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        direct = tgo.moe_layer(hidden, chosen, weights, gate, up, down, *rest)
    torch.cuda.current_stream().wait_stream(side)
    assert not direct.requires_grad and with_gradient.requires_grad
    torch.testing.assert_close(direct, with_gradient.detach(), rtol=0, atol=0)


@pytest.mark.parametrize("shape", ((256,), (3, 512), (2, 3, 40, 256)))
def test_projection_has_the_operators_bits(tgo, shape):
    import synth

    weight = synth.random_packed_weight(QTYPES["Q5_K"], (72,), shape[-1], seed=5).cuda()
    x = random_bf16(shape, seed=6)
    expected = torch.ops.torch_ggml_ops.mmq.default(x, weight, 13, 72)
    assert expected.shape == (*shape[:-1], 72)
    torch.testing.assert_close(tgo.mmq(x, weight, 13, 72), expected, rtol=0, atol=0)


def test_other_calls_reach_the_operator(tgo):
    import synth

    weight = synth.random_packed_weight(12, (64,), 256, seed=7).cuda()
    x = random_bf16((4, 256), seed=8)
    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Watch():
        tgo.mmq(x, weight, 12, 64)
    assert "torch_ggml_ops.mmq.default" in seen
    with torch._subclasses.FakeTensorMode(allow_non_fake_inputs=True) as mode:
        assert tgo.mmq(mode.from_tensor(x), mode.from_tensor(weight), 12, 64).shape == (4, 64)
    with pytest.raises(RuntimeError, match="contiguous"):
        tgo.mmq(x.t().contiguous().t(), weight, 12, 64)
    with pytest.raises(RuntimeError, match="bytes, expected"):
        tgo.mmq(x, weight, 12, 65)
    with pytest.raises(RuntimeError, match="unsupported quant_type"):
        tgo.mmq(x, weight, 1, 64)
    with torch.no_grad():
        assert not tgo.mmq(x.clone().requires_grad_(), weight, 12, 64).requires_grad
    assert tgo.mmq(x.clone().requires_grad_(), weight, 12, 64).requires_grad
