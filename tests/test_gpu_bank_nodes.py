"""The source bank's autograd nodes: which inputs receive a gradient, and what
the nodes keep from one backward call to the next."""

from __future__ import annotations

import math
import operator
import threading

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


def _close(actual, expected):
    """FP32 sums of at most 64 terms in another order (2^-24 of their magnitude each, taken as 2^-18 of the
    largest element), rounded to BF16 for BF16 sources: one unit in the last place, 2^-7 of the element."""
    rtol = 2.0**-7 if expected.dtype == torch.bfloat16 else 2.0**-18
    torch.testing.assert_close(actual.float(), expected.float(), rtol=rtol,
                               atol=2.0**-18 * float(expected.float().abs().max()))


def _full_schedule(sources, queries, gradients="gather", ungraded=()):
    """Push a source, read all so far, over and over; sources whose index is in
    ``ungraded`` are pushed with grad mode off."""
    bank = SourceBank(len(sources), gradients=gradients)
    outs = []
    for i, (source, query) in enumerate(zip(sources, queries)):
        with torch.set_grad_enabled(i not in ungraded):
            bank.push(source)
        outs.append(bank.read(query))
    return outs


def _kept(outs, inputs, grads):
    """The gradients of one pass and the bytes that it leaves allocated besides them."""
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    results = torch.autograd.grad(outs, inputs, grads, retain_graph=True)
    torch.cuda.synchronize()
    return results, torch.cuda.memory_allocated() - before - sum(r.numel() * r.element_size() for r in results)


# 16 reads: slot 7 is the last one with nine of them, the first that may form the sums of slots 6, 5 and 4 too
@pytest.mark.parametrize("ungraded", [(), (0, 1, 2, 3, 4, 5, 6)])
def test_a_pass_forms_no_sums_it_was_not_asked_for(ungraded):
    torch.manual_seed(7)
    tokens, width, reads = 512, 1024, 16
    sources = [_source(tokens, width=width) for _ in range(reads)]
    queries = [_query(width) for _ in range(reads)]
    grads = [torch.randn(tokens, width, device="cuda", dtype=torch.bfloat16) for _ in range(reads)]
    inputs = [sources[7]] if not ungraded else sources[7:]
    results, kept = _kept(_full_schedule(sources, queries, ungraded=ungraded), inputs, grads)
    # the reads' coefficients (12 bytes per source and token) may stay until the next pass; FP32 sums may not
    assert kept < tokens * width * 4, f"{kept} bytes kept"
    expected = torch.autograd.grad(_full_schedule(sources, queries, "accumulate", ungraded), inputs, grads)
    for a, b in zip(results, expected):
        _close(a, b)


class _Streams:
    """Runs pieces of a program on chosen streams, each after all pieces before it."""

    def __init__(self, *streams):
        self.all = (torch.cuda.current_stream(), *streams)

    def run(self, stream, piece):
        for other in self.all:
            if other is not stream:
                stream.wait_stream(other)
        with torch.cuda.stream(stream):
            return piece()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("gradients", ["gather", "accumulate"])
@pytest.mark.parametrize("readers", [1, 2])
def test_pushes_and_reads_on_several_streams(gradients, dtype, readers):
    """Slots 10 to 15 are pushed on one stream, slots 0 to 9 on another and the
    reads run on a third (or a third and a fourth in turn, whose backward kernels
    only the accumulated sums tie together).  In the backward pass the gathers of slots 0 to 9 wait
    behind other work of their stream, long after the pass has let go of the
    reads' terms and of the sums that slot 7's and later gathers
    left for the slots before them; what the other streams allocate and
    overwrite meanwhile must not reach those gathers."""
    torch.manual_seed(8)
    tokens, width, reads, cut = 4096, 256, 16, 10
    sources = [_source(tokens, dtype=dtype, width=width) for _ in range(reads)]
    queries = [_query(width) for _ in range(reads)]
    grads = [torch.randn(tokens, width, device="cuda", dtype=torch.bfloat16) for _ in range(reads)]
    inputs = (*sources, *queries)
    expected = torch.autograd.grad(_full_schedule(sources, queries, gradients), inputs, grads)

    high, low, *reading = (torch.cuda.Stream() for _ in range(2 + readers))
    streams = _Streams(high, low, *reading)
    bank = SourceBank(reads, gradients=gradients)
    outs = []
    for i, (source, query) in enumerate(zip(sources, queries)):
        streams.run(low if i < cut else high, lambda: bank.push(source))
        outs.append(streams.run(reading[i % readers], lambda: bank.read(query)))
    busy = torch.randn(8192, 8192, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(low):  # tens of milliseconds before the low slots' gathers
        for _ in range(5):
            product = busy @ busy
    results = torch.autograd.grad(outs, inputs, grads)
    rubbish = []
    for stream in (high, *reading):
        with torch.cuda.stream(stream):
            for count in range(1, reads + 1):
                rubbish += [torch.empty(3, count, tokens, device="cuda").fill_(float("nan")) for _ in range(2)]
            rubbish += [torch.empty(3, tokens, width, device="cuda").fill_(float("nan")) for _ in range(4)]
            rubbish += [torch.empty(reads, tokens, width, device="cuda").fill_(float("nan")) for _ in range(2)]
    torch.cuda.synchronize()
    del product
    for i, (a, b) in enumerate(zip(results, expected)):
        assert torch.equal(a, b), f"gradient {i}"


@pytest.mark.parametrize("gradients", ["gather", "accumulate"])
def test_nodes_with_saved_tensor_hooks_and_on_another_thread(gradients):
    torch.manual_seed(9)
    sources = [_source(33) for _ in range(12)]
    queries = [_query() for _ in range(12)]
    grads = [torch.randn(33, _WIDTH, device="cuda", dtype=torch.bfloat16) for _ in range(12)]
    inputs = (*sources, *queries)
    expected = torch.autograd.grad(_full_schedule(sources, queries, gradients), inputs, grads)
    with torch.autograd.graph.save_on_cpu():
        outs = _full_schedule(sources, queries, gradients)
    hooked = torch.autograd.grad(outs, inputs, grads)
    outs = _full_schedule(sources, queries, gradients)
    results = []
    thread = threading.Thread(target=lambda: results.extend(torch.autograd.grad(outs, inputs, grads)))
    thread.start()
    thread.join()
    for a, b, c in zip(hooked, results, expected):
        assert torch.equal(a, c) and torch.equal(b, c)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", ["push-all-then-read", "early-reads-of-other-ranks"])
def test_sums_left_for_lower_slots_are_each_slots_own(case, dtype):
    """Slots that get no read after a block formed their sums, and slots whose
    later reads need several launches (two ranks), take the sums as they are or
    add to them; every gradient has memory of its own."""
    torch.manual_seed(10)
    count, tokens = 16, 40
    sources = [_source(tokens, dtype=dtype) for _ in range(count)]
    # slot 7 is the first with nine reads; slots 5 and 4 then get reads 6 and 5 (and 4), of two ranks
    ranks = [_WIDTH // 2 if case.startswith("early") and i in (4, 6) else _WIDTH for i in range(count)]
    queries = [_query(rank) for rank in ranks]
    grads = [torch.randn(tokens, _WIDTH, device="cuda", dtype=torch.bfloat16) for _ in range(count)]

    def outputs(gradients):
        if case.startswith("early"):
            return _full_schedule(sources, queries, gradients)
        bank = SourceBank(count, gradients=gradients)
        for source in sources:
            bank.push(source)
        return [bank.read(query) for query in queries]

    results = torch.autograd.grad(outputs("gather"), sources, grads)
    for a, b in zip(results, torch.autograd.grad(outputs("accumulate"), sources, grads)):
        held, needed = a.untyped_storage().nbytes(), a.numel() * a.element_size()
        assert held == needed
        _close(a, b)
    assert len({a.untyped_storage().data_ptr() for a in results}) == count


@pytest.mark.parametrize("gradients", ["gather", "accumulate"])
def test_a_push_with_grad_mode_off_keeps_the_other_sources_gradients(gradients):
    """Slots 2 and 3 (a push and a sum) are filled with grad mode off: the same
    gradients as with sources that require none."""
    torch.manual_seed(11)
    sources = [_source() for _ in range(6)]
    queries = [_query() for _ in range(6)]

    def outputs(detached):
        bank = SourceBank(6, gradients=gradients)
        outs = []
        for i, (source, query) in enumerate(zip(sources, queries)):
            frozen = source.detach() if detached and i in (2, 3) else source
            with torch.set_grad_enabled(detached or i not in (2, 3)):
                if i == 3:
                    bank.push_sum(frozen, frozen)
                else:
                    bank.push(frozen)
            outs.append(bank.read(query).float().sum())
        return outs

    for reads in ([3], range(6)):  # the read right after them, or all reads
        wanted = [s for i, s in enumerate(sources) if i < 2 or i in reads and i > 3] + [queries[i] for i in reads]
        results = torch.autograd.grad(operator.itemgetter(*reads)(outputs(False)), wanted)
        for a, b in zip(results, torch.autograd.grad(operator.itemgetter(*reads)(outputs(True)), wanted)):
            assert torch.equal(a, b)
