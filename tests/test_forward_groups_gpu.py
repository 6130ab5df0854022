"""Grouped calls with scaled operands whose groups have few rows (run with -m gpu).

Groups of up to 128 rows are handled as one to four tiles of 32 by waves that all unpack and multiply, the others by role-split
workgroups of the same launch; groups of 33 to 128 rows stay with these where they are the fewer.
"""

import numpy as np
import pytest
import torch

from helpers import OPERAND_NOISE, QTYPES, assert_matches_f32_reference, bits, random_bf16

pytestmark = pytest.mark.gpu

SCALE_OFFSETS = {11: (108,), 12: (0, 2), 13: (0, 2), 14: (208,), 22: (0,)}


@pytest.fixture(scope="module")
def ops():
    import synth
    import torch_ggml_ops
    from torch_ggml_ops import _native

    assert torch.cuda.is_available()
    return torch_ggml_ops, _native, synth


@pytest.fixture(autouse=True)
def scaled(ops):
    _, native, _ = ops
    native.set_forward_operand("scaled")
    yield
    native.set_forward_operand("auto")


def _check(ops, oracle, qtype, host, sizes, k, n, pair=False, offset=0):
    tgo, _, _ = ops
    experts = list(range(len(sizes)))[::-1]
    offsets = np.cumsum(sizes).tolist()
    metadata = (torch.tensor(experts, device="cuda"), torch.tensor(offsets, device="cuda", dtype=torch.int32))
    x = random_bf16((offsets[-1], k), seed=offsets[-1] + k)
    flat = torch.zeros(offset + host.numel(), dtype=torch.uint8, device="cuda")
    weight = flat[offset:].view(host.shape)
    weight.copy_(host)
    if pair:
        outputs = tgo.grouped_mmq_pair(x, weight, weight, *metadata, qtype, n)
        assert torch.equal(*outputs)
    else:
        outputs = (tgo.grouped_mmq(x, weight, *metadata, qtype, n),)
    expected = oracle.grouped(oracle.mmq_forward, qtype, bits(x), host.numpy(), experts, offsets, n, k, n)
    assert_matches_f32_reference(outputs[0], expected, OPERAND_NOISE["scaled"])


@pytest.mark.parametrize("qname", tuple(QTYPES))
@pytest.mark.parametrize("k,n", [(256, 264), (768, 200), (2304, 37)])
def test_every_tile_count_and_its_edges(ops, oracle, qname, k, n):
    """1 to 4 row tiles, tasks that start anywhere in a 32-row tile of the workspace, one to nine super-blocks, columns off the tile
    and off the 16-byte stores."""
    qtype = QTYPES[qname]
    sizes = [1, 31, 32, 33, 64, 65, 96, 97, 128, 129] + [1] * 20
    host = ops[2].random_packed_weight(qtype, (len(sizes), n), k, seed=qtype + k)
    _check(ops, oracle, qtype, host, sizes, k, n, pair=n == 200)


@pytest.mark.parametrize("qname", ("Q3_K", "Q6_K", "IQ2_S"))
def test_weights_whose_experts_do_not_start_on_16_bytes(ops, oracle, qname):
    """An odd number of weight rows: bytes per expert are no multiple of 16, and the packed blocks are copied two bytes at a time."""
    qtype = QTYPES[qname]
    sizes = [40, 3, 100]
    host = ops[2].random_packed_weight(qtype, (len(sizes), 133), 256, seed=qtype)
    _check(ops, oracle, qtype, host, sizes, 256, 133)


@pytest.mark.parametrize("qname", tuple(QTYPES))
def test_super_blocks_of_very_different_size(ops, oracle, qname):
    """A weight row's normalisation follows its super-blocks: scales that grow by up to 2^12 from one super-block to the next, shrink,
    or are zero at first, in different rows at different places."""
    qtype, k, n, sizes = QTYPES[qname], 2048, 96, [5, 70, 33, 128]
    host = ops[2].random_packed_weight(qtype, (len(sizes), n), k, seed=5)
    blocks = host.view(len(sizes), n, k // 256, -1)
    rng = np.random.default_rng(qtype)
    power = rng.choice([-9, -7, -3, 0, 3], size=(len(sizes), n, k // 256)).astype(np.float32)
    power[:, ::3] = np.linspace(-9, 3, k // 256)          # growing all the way
    factor = torch.from_numpy(np.exp2(power).astype(np.float16))
    factor[:, 1::3, 0] = 0.0
    for offset in SCALE_OFFSETS[qtype]:
        scale = blocks[..., offset : offset + 2].contiguous().view(torch.float16)[..., 0]
        blocks[..., offset : offset + 2] = (scale * factor).view(torch.uint8).view(*factor.shape, 2)
    _check(ops, oracle, qtype, host, sizes, k, n)


@pytest.mark.parametrize("k", (512, 1024))
@pytest.mark.parametrize("sizes", ([700, 20, 513, 5], [1000, 300, 33, 1], [280, 40, 60, 130], [140, 140, 40, 200], [256, 150, 30, 4], [32, 1, 7]))
def test_lists_with_more_and_with_fewer_small_groups(ops, oracle, k, sizes):
    """More and fewer groups of 33 to 128 rows than larger tasks, none of them, and only the smallest."""
    qtype, n = QTYPES["Q5_K"], 200
    host = ops[2].random_packed_weight(qtype, (len(sizes), n), k, seed=7)
    _check(ops, oracle, qtype, host, sizes, k, n)


def test_more_groups_than_one_round_of_the_list_builder(ops, oracle):
    """The list is built 256 groups at a time: 600 groups of every class in no order."""
    qtype, k, n = QTYPES["Q4_K"], 256, 32
    rng = np.random.default_rng(1)
    sizes = rng.choice([0, 1, 3, 30, 33, 50, 130], size=600, p=[0.1, 0.4, 0.2, 0.1, 0.1, 0.07, 0.03]).tolist()
    host = ops[2].random_packed_weight(qtype, (len(sizes), n), k, seed=9)
    _check(ops, oracle, qtype, host, sizes, k, n)


def _spread_weights(ops, qtype, experts, n, k, power):
    """Random packed weights whose super-block s has scales 2^power[s] times those of a usual one."""
    host = ops[2].random_packed_weight(qtype, (experts, n), k, seed=qtype)
    blocks = host.view(experts, n, k // 256, -1)
    factor = torch.exp2(torch.tensor(power, dtype=torch.float32)).expand(experts, n, k // 256)
    for offset in SCALE_OFFSETS[qtype]:
        scale = blocks[..., offset : offset + 2].contiguous().view(torch.float16)[..., 0].float()
        blocks[..., offset : offset + 2] = (scale * factor).to(torch.float16).contiguous().view(torch.uint8).view(*factor.shape, 2)
    return host


@pytest.mark.parametrize("qname", tuple(QTYPES))
@pytest.mark.parametrize("largest_first", (True, False))
def test_up_to_32_rows_every_super_block_keeps_its_own_bits(ops, oracle, qname, largest_first):
    """Weights 2^18 below another super-block of their row, which meets activations of zero: the result is theirs alone, and as
    exact as if the other were not there."""
    tgo, _, _ = ops
    qtype, k, n, sizes = QTYPES[qname], 768, 96, [1, 20, 32]
    power = [9, -9, -9] if largest_first else [-9, -9, 9]
    host = _spread_weights(ops, qtype, len(sizes), n, k, power)
    offsets = np.cumsum(sizes).tolist()
    x = random_bf16((offsets[-1], k), seed=3)
    x[:, :256] = 0 if largest_first else x[:, :256]
    x[:, 512:] = 0 if not largest_first else x[:, 512:]
    metadata = (torch.arange(len(sizes), device="cuda"), torch.tensor(offsets, device="cuda", dtype=torch.int32))
    output = tgo.grouped_mmq(x, host.cuda(), *metadata, qtype, n)
    expected = oracle.grouped(oracle.mmq_forward, qtype, bits(x), host.numpy(), list(range(len(sizes))), offsets, n, k, n)
    assert_matches_f32_reference(output, expected, OPERAND_NOISE["scaled"])


@pytest.mark.parametrize("qname", tuple(QTYPES))
def test_33_to_128_rows_are_as_exact_as_a_dense_call(ops, qname):
    """With the row's largest super-block first, the weights are normalised as in the role-split kernel of a dense call, also those
    that lose bits: the same results bit for bit.  2^14 and 2^20 below the largest, at which the activations are small."""
    tgo, _, _ = ops
    qtype, k, n, sizes = QTYPES[qname], 768, 96, [33, 64, 70, 96, 100, 128]
    host = _spread_weights(ops, qtype, len(sizes), n, k, [9, -5, -11]).cuda()
    offsets = np.cumsum(sizes).tolist()
    x = random_bf16((offsets[-1], k), seed=4)
    x[:, :256] *= 2.0**-20
    metadata = (torch.arange(len(sizes), device="cuda"), torch.tensor(offsets, device="cuda", dtype=torch.int32))
    output = tgo.grouped_mmq(x, host, *metadata, qtype, n)
    for expert, (begin, end) in enumerate(zip([0] + offsets, offsets)):
        dense = tgo.mmq(x[begin:end].clone(), host[expert].clone(), qtype, n)
        torch.testing.assert_close(output[begin:end], dense, rtol=0, atol=0)
