"""Reads of few tokens run one workgroup per token (attnres_fwd_few_kernel);
reads of many stream their tokens.  A token's output, refinement bytes and
saved statistics are the same bits either way, so a decoded token matches the
same token of a prefill."""

from __future__ import annotations

import math

import pytest
import torch

from attnres import _ops

pytestmark = pytest.mark.gpu

_MANY = 9000  # tokens: past the few-token range of every width and source count


@pytest.mark.parametrize("layout", ["packed", "list"])
@pytest.mark.parametrize("sources,width,rank,offset", [
    # every geometry, whole and partial rows, with and without key masks, aligned or not
    (1, 64, 64, 0), (2, 128, 128, 0), (129, 104, 30, 0), (7, 5, 5, 0), (3, 1, 1, 0), (30, 9, 4, 0),
    (25, 256, 256, 0), (12, 129, 129, 0), (49, 200, 64, 1),
    (25, 512, 128, 0), (33, 511, 511, 0), (64, 1024, 1024, 0), (8, 1024, 256, 0), (17, 770, 769, 0), (5, 768, 768, 1),
    (25, 2048, 2048, 0), (49, 2048, 512, 0), (16, 1536, 1536, 0), (13, 1537, 385, 0), (2, 2047, 2047, 0),
    (25, 4096, 4096, 0), (9, 4096, 1024, 0), (18, 3000, 3000, 1), (129, 2049, 2000, 0),
    (9, 8192, 8192, 0), (25, 5120, 1280, 0), (6, 4097, 4097, 0), (3, 8191, 100, 0),
])
def test_few_tokens_equal_the_same_tokens_of_a_large_read(sources, width, rank, offset, layout):
    print(f"few tokens S={sources} D={width} R={rank} offset={offset} {layout}", flush=True)
    many = max(1200, min(_MANY, 300_000_000 // (sources * width)))
    torch.manual_seed(sources + width)
    values = torch.randn(sources, many, width + offset, device="cuda", dtype=torch.bfloat16)[..., offset:]
    values = values * torch.linspace(0.5, 4, sources, device="cuda", dtype=torch.bfloat16)[:, None, None] \
        if offset == 0 else values
    query = (torch.randn(rank, device="cuda") * 3 / math.sqrt(rank)).to(torch.bfloat16)

    def forward(rows):
        if layout == "packed":
            return _ops.packed_forward_impl(rows, query, 2**-23, 1.0, True)
        return _ops.sources_forward_impl(list(rows.unbind(0)), query, 2**-23, 1.0, True)

    whole = forward(values)
    for count in (1, 3, 40):
        few = forward(values[:, :count])
        torch.cuda.synchronize()
        for name, a, b in zip(("out", "refine", "logit", "inv_rms"), few, whole):
            assert torch.equal(a, b[:count]), f"{name} of {count} tokens"
        assert torch.equal(few[4], whole[4][:, :count]), f"stats of {count} tokens"


@pytest.mark.parametrize("width", [1024, 2048, 4097])
def test_few_tokens_with_special_values(width):
    """Infinite and NaN rows, and logits that overflow, give what the same
    tokens of a large read give (NaN in the same places)."""
    sources, many = 9, 4000
    torch.manual_seed(3)
    values = torch.randn(sources, many, width, device="cuda", dtype=torch.bfloat16)
    values[2, 0, 5] = float("inf")
    values[4, 1, width - 1] = float("nan")
    values[0, 2] = float("nan")
    values[:, 3] = 0
    values[8, 4] = 3e38
    query = torch.randn(width, device="cuda").to(torch.bfloat16)
    for scale in (1.0, 1e30, -1e30):
        whole = _ops.packed_forward_impl(values, query, 2**-23, scale, True)
        few = [_ops.packed_forward_impl(values[:, n:n + 1], query, 2**-23, scale, True) for n in range(6)]
        torch.cuda.synchronize()
        for n, one in enumerate(few):
            torch.testing.assert_close(one[2], whole[2][n:n + 1], rtol=0, atol=0, equal_nan=True)
            torch.testing.assert_close(one[0], whole[0][n:n + 1], rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("sources,width", [(3, 256), (4, 256), (2, 64), (8, 1536), (9, 1536), (8, 1025), (9, 1025), (2, 2048)])
def test_both_sides_of_one_and_two_tokens_per_cu(sources, width):
    """Whether a few tokens' read runs one workgroup per token also depends on
    its width and sources: around 256 and 512 tokens (a CU each, two) the bits
    are those of the same tokens of a large read."""
    torch.manual_seed(sources + width)
    values = torch.randn(sources, 3000, width, device="cuda", dtype=torch.bfloat16)
    query = (torch.randn(width, device="cuda") * 3 / math.sqrt(width)).to(torch.bfloat16)
    whole = _ops.packed_forward_impl(values, query, 2**-23, 1.0, True)
    for count in (256, 257, 512, 513):
        few = _ops.packed_forward_impl(values[:, :count], query, 2**-23, 1.0, True)
        torch.cuda.synchronize()
        for a, b in zip(few[:4], whole):
            assert torch.equal(a, b[:count])
        assert torch.equal(few[4], whole[4][:, :count])
