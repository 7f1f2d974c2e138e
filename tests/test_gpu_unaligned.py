"""Rows that no 16-byte access is aligned to, against the CPU oracle.

Such rows take 16-byte accesses at element alignment, and a width that is no
multiple of 8 ends in a chunk moved back over the chunk before it.  The
widths here put that last chunk everywhere it can go wrong: every remainder
of 8, the first and the last lane of a chunk column, the first lane of a
second column and of another wavefront, and rows too short to hold one chunk.
"""

from __future__ import annotations

import math

import pytest
import torch

from attnres import SharedSources, SourceBank, attnres
from helpers import both_oracles, check_statistics, compare_read, set_case

pytestmark = pytest.mark.gpu

_REMAINDERS = [1, 5, 7, 8, 9, 10, 11, 12, 13, 14, 15]
_COLUMNS = [127, 129, 257, 263, 505, 513, 769, 1025, 1530, 1537, 2047, 2049, 2563, 3073, 4094, 4097, 5121, 6145, 8187]


def _leaves(sources, tokens, width, offset, rank):
    torch.manual_seed(width + sources)
    producer = torch.randn(sources, tokens, width + offset, device="cuda", dtype=torch.bfloat16).requires_grad_()
    query = (torch.randn(rank, device="cuda") / math.sqrt(rank)).to(torch.bfloat16).requires_grad_()
    upstream = torch.randn(tokens, width, device="cuda", dtype=torch.bfloat16)
    return producer, query, upstream


@pytest.mark.parametrize("sources", [3, 14])
@pytest.mark.parametrize("width,offset", [(w, 0) for w in _REMAINDERS + _COLUMNS] +
                         [(w, 1) for w in (8, 128, 512, 1024, 2048, 4096, 8192)])
def test_unaligned_rows_match_oracle(width, offset, sources):
    rank = width if width % 2 else max(1, width // 3)
    tokens = 5 if width > 2048 else 19
    print(f"unaligned S={sources} N={tokens} D={width} R={rank} offset={offset}", flush=True)
    producer, query, upstream = _leaves(sources, tokens, width, offset, rank)

    def make(leaves, q):
        return leaves[0][..., offset:], q

    set_case(f"unaligned S={sources} D={width} R={rank} offset={offset}")
    out = attnres(make([producer], query)[0], query)
    grads = torch.autograd.grad(out, (producer, query), upstream)
    expected, exact = both_oracles(make, [producer], query, upstream)
    torch.cuda.synchronize()
    compare_read((out, *grads), expected, exact, ["out", "dv", "dq"], sources=sources)
    check_statistics(make([producer.detach()], query)[0], query.detach())


@pytest.mark.parametrize("width", [7, 9, 263, 513, 1025, 2049, 4097])
def test_summed_gradients_of_unaligned_rows(width):
    """The accumulating (BF16 and FP32) and the gathered source gradients add
    each element once, also where the row's last two chunks overlap: the sum
    over two equal reads is twice one read's gradient.  The BF16 sums are that
    exactly (bf16(v) + v lies within half a unit of 2 bf16(v), whose spacing is
    two); the FP32 sums up to one BF16 rounding and, where an element's terms
    cancel, the FP32 rounding of a dozen terms of the gradient's size (2^-20
    of its maximum)."""
    sources, tokens = 8, 11
    print(f"unaligned sums D={width}", flush=True)
    producer, query, upstream = _leaves(sources, tokens, width, 0, width)
    rows = [r.detach().clone().requires_grad_() for r in producer]

    shared = SharedSources(rows)
    once = torch.autograd.grad(shared.read(query), rows, upstream)
    shared = SharedSources(rows)
    twice = torch.autograd.grad([shared.read(query), shared.read(query)], rows, [upstream, upstream])
    for one, two in zip(once, twice):
        assert torch.equal(two, 2 * one)
    for gradients in ("gather", "accumulate"):
        def bank_grads(reads):
            bank = SourceBank(sources, gradients=gradients)
            for row in rows:
                bank.push(row)
            return torch.autograd.grad([bank.read(query) for _ in range(reads)], rows, [upstream] * reads)

        for one, two in zip(bank_grads(1), bank_grads(2)):
            atol = 2.0**-20 * float(one.float().abs().max())
            torch.testing.assert_close(two.float(), 2 * one.float(), rtol=2.0**-7, atol=atol)
            # one read's gradient is the plain read's up to a BF16 rounding
        plain = torch.autograd.grad(attnres(tuple(rows), query), rows, upstream)
        for one, ref in zip(bank_grads(1), plain):
            scale = float(ref.float().abs().max())
            torch.testing.assert_close(one.float(), ref.float(), rtol=2.0**-7, atol=2.0**-12 * scale)
