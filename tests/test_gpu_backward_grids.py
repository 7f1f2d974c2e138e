"""The grids of the backward kernels of 3-chunk rows (513-768, 1025-1536 and
4097-6144 elements) depend on how many tokens each group would take.  dq, which
every workgroup adds a partial row to, on both sides of each line of the rule,
against float64."""

from __future__ import annotations

import math

import pytest
import torch

from attnres import attnres

pytestmark = pytest.mark.gpu


def _exact_dq(values, query, grad):
    """dq and the size its FP32 terms' errors are relative to (every product of the
    inner sums taken by magnitude), float64, in token chunks."""
    sources, tokens, width = values.shape
    rank = query.numel()
    q = query.double()
    dq = torch.zeros(rank, device="cuda", dtype=torch.float64)
    size = torch.zeros_like(dq)
    for at in torch.arange(tokens, device="cuda").split(1024):
        v, g = values[:, at].double(), grad[at].double()
        key = v[..., width - rank:]
        inv_rms = torch.rsqrt(key.square().mean(-1) + 2**-23)
        p = ((key @ q) * inv_rms).softmax(0)
        dw, dw_size = (v * g).sum(-1), (v * g).abs().sum(-1)
        a = p * (dw - (p * dw).sum(0)) * inv_rms
        a_size = p * (dw_size + (p * dw_size).sum(0)) * inv_rms
        dq += (a[..., None] * key).sum((0, 1))
        size += (a_size[..., None] * key.abs()).sum((0, 1))
    return dq, size


# tokens of one, two and four rounds of the grids (8, 4 or 1 groups per workgroup, one or two workgroups per CU of 256)
_EDGES = [(w, r, pad, n) for w, r, pad, f in ((768, 192, 0, 8), (600, 600, 1, 8), (1536, 1536, 0, 4), (1025, 300, 0, 4),
                                             (6144, 6144, 0, 1), (5120, 1280, 0, 1), (4099, 4099, 1, 1))
          for n in (512 * f - 1, 512 * f, 1024 * f - 1, 1024 * f, 1024 * f + 1, 1100 * f)]


@pytest.mark.parametrize("sources", [2, 7])
@pytest.mark.parametrize("width,rank,pad,tokens", _EDGES)
def test_query_gradient_at_the_edges_of_the_grids(width, rank, pad, tokens, sources):
    print(f"backward grid D={width} R={rank} pad={pad} N={tokens} S={sources}", flush=True)
    torch.manual_seed(width + tokens)
    values = torch.randn(sources, tokens, width + pad, device="cuda", dtype=torch.bfloat16)[..., pad:].requires_grad_()
    query = (torch.randn(rank, device="cuda") / math.sqrt(rank)).to(torch.bfloat16).requires_grad_()
    grad = torch.randn(tokens, width, device="cuda", dtype=torch.bfloat16)
    (dq,) = torch.autograd.grad(attnres(values, query), query, grad)
    exact, size = _exact_dq(values.detach(), query.detach(), grad)
    # the result's BF16 rounding (half a unit: 2^-9), and FP32 sums: a lane adds at most 24 products of a row before
    # the lanes meet in 8 steps, so dw, delta and the norm are off by at most 32 * 2^-24 of their terms' magnitude
    bound = 2.0**-9 * exact.abs() + 2.0**-19 * size
    assert bool(((dq.double() - exact).abs() <= bound).all())
