"""A source bank's slot with many reads forms the FP32 sums of the slots
before it too (one pass over the dO rows they share); those slots add their
later reads to them.  Against the accumulating gradients (FP32 sums of every
read's dv, formed in another kernel): the two differ by the rounding of FP32
sums of about 2 * reads terms, 2^-24 of their magnitude each, taken here as
2^-18 of the gradient's largest element; where the source is BF16 such a
difference can also turn a rounding, by one unit in the last place, which is at
most 2^-7 of the element."""

from __future__ import annotations

import math

import pytest
import torch

from attnres import SourceBank

pytestmark = pytest.mark.gpu


def _case(width, rank, reads, tokens, dtype):
    torch.manual_seed(width + reads)
    sources = [torch.randn(2, tokens, width, device="cuda", dtype=dtype).requires_grad_() for _ in range(reads)]
    queries = [(torch.randn(rank, device="cuda") / math.sqrt(rank)).to(torch.bfloat16).requires_grad_()
               for _ in range(reads)]
    grads = [torch.randn(2, tokens, width, device="cuda", dtype=torch.bfloat16) for _ in range(reads)]
    return sources, queries, grads


def _outputs(sources, queries, gradients):
    bank = SourceBank(len(sources), gradients=gradients)
    outs = []
    for source, query in zip(sources, queries):
        bank.push(source)
        outs.append(bank.read(query))
    return outs


def _close(actual, expected, dtype):
    atol = 2.0**-18 * float(expected.float().abs().max())
    rtol = 2.0**-7 if dtype == torch.bfloat16 else 2.0**-18
    torch.testing.assert_close(actual.float(), expected.float(), rtol=rtol, atol=atol)


_SHAPES = [(64, 64), (200, 50), (256, 256), (512, 512), (640, 160), (1024, 1024), (1025, 1025), (1472, 1472),
           (2048, 512), (2560, 2560), (4096, 1024), (5000, 5000), (8191, 8191)]


# 8: no block; 9: the first block at its smallest; 12 and 13: whole and uneven blocks; 52: more reads than a launch
# (a narrow, a wide and an unaligned row)
@pytest.mark.parametrize("width,rank,reads", [(w, r, n) for w, r in _SHAPES for n in (8, 9, 12, 13, 21)] +
                         [(w, w, 52) for w in (64, 1024, 1025)])
def test_blocks_of_slots_match_accumulated_gradients(width, rank, reads):
    dtype = torch.bfloat16 if reads % 2 else torch.float32
    print(f"bank blocks D={width} R={rank} reads={reads} {dtype}", flush=True)
    sources, queries, grads = _case(width, rank, reads, 9 if width > 1024 else 37, dtype)
    gathered = torch.autograd.grad(_outputs(sources, queries, "gather"), (*sources, *queries), grads)
    summed = torch.autograd.grad(_outputs(sources, queries, "accumulate"), (*sources, *queries), grads)
    for a, b in zip(gathered[:reads], summed[:reads]):
        _close(a, b, dtype)
    for a, b in zip(gathered[reads:], summed[reads:]):
        torch.testing.assert_close(a, b, rtol=2.0**-7, atol=2.0**-12 * float(b.float().abs().max()))


def test_blocks_with_frozen_sources_and_partial_passes():
    """Slots without a gradient break the blocks; a pass that asks for some
    sources only, and a second pass over the same graph, give the same bits."""
    sources, queries, grads = _case(1024, 1024, 16, 40, torch.float32)
    whole = torch.autograd.grad(_outputs(sources, queries, "gather"), sources, grads)
    outs = _outputs(sources, queries, "gather")
    some = [sources[i] for i in (12, 6, 5, 0)]
    part = torch.autograd.grad(outs, some, grads, retain_graph=True)
    again = torch.autograd.grad(outs, sources, grads)
    for a, b in zip(part, (whole[12], whole[6], whole[5], whole[0])):
        _close(a, b, torch.float32)
    for a, b in zip(again, whole):
        assert torch.equal(a, b)
    frozen = [s.detach().requires_grad_(i not in (3, 6)) for i, s in enumerate(sources)]
    wanted = [s for s in frozen if s.requires_grad]
    result = torch.autograd.grad(_outputs(frozen, queries, "gather"), wanted, grads)
    for a, b in zip(result, [g for i, g in enumerate(whole) if i not in (3, 6)]):
        _close(a, b, torch.float32)
