"""The source bank's autograd nodes: which inputs receive a gradient, and what
the nodes keep from one backward call to the next."""

from __future__ import annotations

import math

import pytest
import torch

from attnres import SourceBank

pytestmark = pytest.mark.gpu

_WIDTH = 64


def _source(tokens=10, dtype=torch.float32, width=_WIDTH):
    return torch.randn(tokens, width, device="cuda", dtype=dtype).requires_grad_()


def _query(width=_WIDTH):
    return (torch.randn(width, device="cuda") / math.sqrt(width)).to(torch.bfloat16).requires_grad_()


class _Absent(torch.autograd.Function):
    """Passes a value on and gives no gradient for it."""

    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, _grad):
        return None


@pytest.mark.parametrize("gradients", ["gather", "accumulate"])
def test_an_unused_partial_sum_gives_zero_gradients(gradients):
    """Neither the sum nor its slot is used after push_sum: its inputs get
    zeros, also where autograd is asked for them by name."""
    torch.manual_seed(5)
    first, prev, emitted, query = _source(), _source(), _source(), _query()
    bank = SourceBank(4, gradients=gradients)
    bank.push(first, slot=0)
    bank.push_sum(prev, emitted, slot=2)
    out = bank.read(query, count=1)
    grads = torch.autograd.grad(out.float().sum(), [first, prev, emitted, query])
    assert torch.equal(grads[0], torch.ones_like(first))
    assert grads[1].dtype == prev.dtype and torch.equal(grads[1], torch.zeros_like(prev))
    assert torch.equal(grads[2], torch.zeros_like(emitted))


@pytest.mark.parametrize("gradients", ["gather", "accumulate"])
def test_a_read_without_an_upstream_gradient_gives_zero_gradients(gradients):
    torch.manual_seed(6)
    source, later, query, query2 = _source(), _source(), _query(), _query()
    bank = SourceBank(4, gradients=gradients)
    bank.push(source)
    only = bank.read(query)
    grads = torch.autograd.grad(_Absent.apply(only).float().sum(), [source, query], retain_graph=True)
    assert torch.equal(grads[0], torch.zeros_like(source)) and torch.equal(grads[1], torch.zeros_like(query))
    bank.push(later)
    second = bank.read(query2)
    loss = _Absent.apply(only).float().sum() + second.float().sum()
    grads = torch.autograd.grad(loss, [source, later, query, query2], retain_graph=True)
    assert torch.equal(grads[2], torch.zeros_like(query))
    expected = torch.autograd.grad(second.float().sum(), [source, later, query2])
    for a, b in zip((grads[0], grads[1], grads[3]), expected):
        assert torch.equal(a, b)
