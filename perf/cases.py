"""Timed workloads of the attnres read, from one decoded token to a deep training read.

`listed()` names the workloads, `draw()` gives more of the same ranges, and
`prepare` / `run` hold what a program has before a pass and the pass itself,
through the package's public entry points:

* ``read``:   forward and backward of ``attnres`` on packed ``[S, B, T, D]`` values;
* ``list``:   the same on an ordered list of S separate ``[B, T, D]`` tensors;
* ``infer``:  the forward alone (``torch.no_grad``) on packed values;
* ``decode``: one decoding step of a Full-schedule model, reads of 1..S sources
  of a few tokens, captured once in a HIP graph and replayed per step, as a
  serving loop does with its launch-bound steps;
* ``bank``:   a Full-schedule pass through ``SourceBank``: push a source, read
  all sources so far, S times over, then one backward pass through all of it.

Values have a standard deviation of 0.5 to 4 per source and 1% of channels
eight times larger; queries are N(0, 1) / sqrt(R), upstream gradients N(0, 1).
"""

from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parents[1] / "fast-attnres_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from attnres import SourceBank, attnres  # noqa: E402

_EPS = 2**-23
_MAX_VALUES = 1_600_000_000  # elements of a drawn case's values; the largest listed case has twice as many


def _case(kind: str, sources: int, batch: int, tokens: int, width: int, rank: int, *, pad: int = 0, **name) -> dict:
    return {**name, "kind": kind, "sources": sources, "batch": batch, "tokens": tokens, "width": width, "rank": rank,
            "pad": pad}


def listed() -> list[dict]:
    return [
        # one token of one sequence, eagerly: the shortest call there is
        _case("infer", 25, 1, 1, 2048, 2048, name="infer-one-token"),
        # a decoding step of the 24-layer, 1024-wide model for 16 sequences: 48 reads in one graph
        _case("decode", 48, 16, 1, 1024, 1024, name="decode-step-24-layers"),
        # the small read of the CPU configuration, two sequences of 512 tokens
        _case("read", 8, 2, 512, 1024, 1024, name="train-small"),
        # a middle read of the 24-layer training workload, 2 x 1024 tokens
        _case("read", 25, 2, 1024, 1024, 1024, name="train-2k-tokens"),
        # prefill of one long prompt
        _case("infer", 25, 1, 4096, 2048, 2048, name="infer-prefill"),
        # odd sizes all round: no power of two, rows that no wide load is aligned to
        _case("read", 13, 3, 1365, 1537, 385, name="train-ragged"),
        # the headline read: 25 sources, 16384 tokens
        _case("read", 25, 8, 2048, 2048, 2048, name="train-headline"),
        # low-rank routing: the key is the last quarter of the row
        _case("read", 16, 1, 16384, 4096, 1024, name="train-low-rank"),
        # a wide row between the powers of two
        _case("read", 17, 2, 4096, 5120, 1280, name="train-wide"),
        # Block schedule: eight block sums and the embedding, separate tensors
        _case("list", 9, 1, 32768, 2048, 2048, name="train-block-list"),
        # the residual stream of a Full-schedule model, 16 x 1024 tokens
        _case("bank", 20, 16, 1024, 1024, 1024, name="bank-full-schedule"),
        # the last read of a 24-layer, 4096-wide model: the largest
        _case("read", 48, 8, 2048, 4096, 4096, name="train-deep"),
    ]


def _log_uniform(rng: random.Random, low: int, high: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _width(rng: random.Random, high: int) -> int:
    width = _log_uniform(rng, 256, high)
    step = rng.choice((256, 256, 128, 8, 8, 1))  # most rows are round, some are not
    return max(step, width // step * step)


def _rank(rng: random.Random, width: int) -> int:
    return rng.choice((width, width, width, width // 4, width // 4, rng.randint(1, width)))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(("read",) * 6 + ("list",) * 3 + ("infer",) * 4 + ("decode",) * 3 + ("bank",) * 3)
    if kind == "decode":
        width = _width(rng, 4096)
        return _case(kind, rng.randint(8, 48), _log_uniform(rng, 1, 64), 1, width, _rank(rng, width))
    if kind == "bank":
        width = _log_uniform(rng, 256, 2048) // 64 * 64
        sources = rng.randint(4, 20)
        tokens = min(_log_uniform(rng, 256, 16384), 400 * 16384 * 1024 // (sources * sources * width))
        batch = rng.randint(1, 4)
        return _case(kind, sources, batch, tokens // batch, width, rng.choice((width, width // 4)))
    width = _width(rng, 8192)
    sources = _log_uniform(rng, 1, 49)
    tokens = _log_uniform(rng, 1 if kind == "infer" else 256, 32768)
    tokens = max(1, min(tokens, _MAX_VALUES // (sources * width)))
    batch = rng.choice((1, 1, rng.randint(1, 8)))
    batch = min(batch, tokens)
    # values of a padded producer: rows further apart than they are wide
    pad = rng.choice((0, 0, 0, 8, 1)) if kind != "list" else 0
    return _case(kind, sources, batch, max(1, tokens // batch), width, _rank(rng, width), pad=pad)


# ------------------------------------------------------------------- inputs


def _inputs(case: dict, seed: int):
    """values [S, B, T, D], queries (one, or one per read) and upstream gradients."""
    device = torch.device("cuda")
    generator = torch.Generator(device=device).manual_seed(seed)
    sources, width, rank = case["sources"], case["width"], case["rank"]
    shape = (case["batch"], case["tokens"], width)
    std = torch.rand(sources, generator=generator, device=device) * 3.5 + 0.5
    scale = torch.ones(width, device=device)
    scale[torch.randperm(width, generator=generator, device=device)[: max(1, width // 100)]] = 8.0
    buffer = torch.empty((sources, *shape[:2], width + case["pad"]), device=device, dtype=torch.bfloat16)
    values = buffer[..., case["pad"]:]
    for s in range(sources):
        values[s] = torch.randn(shape, generator=generator, device=device) * (std[s] * scale)
    many = sources if case["kind"] in ("decode", "bank") else 1
    queries = [(torch.randn(rank, generator=generator, device=device) / math.sqrt(rank)).to(torch.bfloat16)
               for _ in range(many)]
    backward = case["kind"] in ("read", "list", "bank")
    grads = [torch.randn(shape, generator=generator, device=device).to(torch.bfloat16)
             for _ in range(many if backward else 0)]
    return values, queries, grads


def _decode_step(values, queries) -> list[torch.Tensor]:
    with torch.no_grad():
        return [attnres(values[: i + 1], query) for i, query in enumerate(queries)]


def prepare(case: dict, seed: int) -> dict:
    values, queries, grads = _inputs(case, seed)
    kind = case["kind"]
    state = {"kind": kind, "values": values, "queries": queries, "grads": grads}
    if kind == "decode":
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):  # once outside the capture
            _decode_step(values, queries)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state["outputs"] = _decode_step(values, queries)
        state["graph"] = graph
    elif kind in ("list", "bank"):
        state["sources"] = [v.clone().requires_grad_(True) for v in values]
        state["values"] = None
    elif kind == "read":
        state["values"] = values.detach().requires_grad_(True)
    if grads:
        state["queries"] = [q.requires_grad_(True) for q in queries]
    return state


def run(state: dict):
    kind = state["kind"]
    if kind == "decode":
        state["graph"].replay()
        return state["outputs"]
    if kind == "infer":
        with torch.no_grad():
            return attnres(state["values"], state["queries"][0])
    if kind == "bank":
        bank = SourceBank(capacity=len(state["sources"]))
        outs = []
        for source, query in zip(state["sources"], state["queries"]):
            bank.push(source)
            outs.append(bank.read(query))
        grads = torch.autograd.grad(outs, [*state["sources"], *state["queries"]], state["grads"])
        count = len(outs)
        return {"out": [out.detach() for out in outs], "dv": list(grads[:count]), "dq": list(grads[count:])}
    query, upstream = state["queries"][0], state["grads"][0]
    if kind == "list":
        out = attnres(state["sources"], query)
        *dv, dq = torch.autograd.grad(out, [*state["sources"], query], upstream)
        return {"out": out.detach(), "dv": dv, "dq": dq}
    out = attnres(state["values"], query)
    dv, dq = torch.autograd.grad(out, (state["values"], query), upstream)
    return {"out": out.detach(), "dv": dv, "dq": dq}


# ------------------------------------------------- what a pass cannot do without


def work(case: dict) -> dict:
    """Bytes: a forward reads its values and writes its output; a backward
    reads the values and the upstream gradient and writes the value
    gradients (a bank writes one gradient per source for all its reads)."""
    sources, rank = case["sources"], case["rank"]
    elements = case["batch"] * case["tokens"] * case["width"]
    keys = case["batch"] * case["tokens"] * rank
    kind = case["kind"]
    reads = sources * (sources + 1) // 2 if kind in ("decode", "bank") else sources  # source rows read forward
    outs = sources if kind in ("decode", "bank") else 1
    rows, flops = reads + outs, reads * (2 * elements + 4 * keys)
    if kind in ("read", "list", "bank"):
        rows += reads + outs + sources
        flops += reads * (4 * elements + 6 * keys)
    if kind == "bank":
        rows += 2 * sources  # each pushed source is read and stored in its slot
    return {"bytes": 2 * rows * elements, "flops": flops}


def tolerance(case: dict) -> dict:
    """BF16 results of FP32 arithmetic, rounded once: an implementation is off
    the exact value by a relative 1.7e-3 (every element within half a unit in
    the last place, 2^-9), and a single element by up to 2^-8 of itself; four
    times that."""
    return {"rel": 7e-3, "max": 2**-6}


# -------------------------------------------------------------------- 64 bits


def _exact_read(values, query, upstream):
    """out, dv, dq of one read in float64, token chunk by token chunk."""
    sources, width = values.shape[0], values.shape[-1]
    rank = query.numel()
    flat = values.detach().reshape(sources, -1, width)
    tokens = flat.shape[1]
    q = query.detach().double()
    out = torch.empty((tokens, width), device=flat.device, dtype=torch.float64)
    dv = dq = g_rows = None
    if upstream is not None:
        dv = torch.empty((sources, tokens, width), device=flat.device, dtype=torch.float64)
        dq = torch.zeros(rank, device=flat.device, dtype=torch.float64)
        g_rows = upstream.reshape(-1, width)
    step = max(1, 200_000_000 // (sources * width))
    for first in range(0, tokens, step):
        at = slice(first, min(tokens, first + step))
        v = flat[:, at].double()
        key = v[..., width - rank:]
        inv_rms = torch.rsqrt(key.square().mean(-1) + _EPS)
        z = (key @ q) * inv_rms
        p = z.softmax(0)
        out[at] = (p[..., None] * v).sum(0)
        if upstream is None:
            continue
        g = g_rows[at].double()
        dw = (v * g).sum(-1)
        dz = p * (dw - (p * dw).sum(0))
        a = dz * inv_rms
        part = p[..., None] * g
        part[..., width - rank:] += a[..., None] * q - (a * inv_rms * z / rank)[..., None] * key
        dv[:, at] = part
        dq += (a[..., None] * key).sum((0, 1))
    shape = values.shape[1:]
    return out.reshape(shape), None if dv is None else dv.reshape(values.shape), dq


def exact(case: dict, seed: int):
    values, queries, grads = _inputs(case, seed)
    kind = case["kind"]
    if kind == "infer":
        return _exact_read(values, queries[0], None)[0]
    if kind == "decode":
        return [_exact_read(values[: i + 1], query, None)[0] for i, query in enumerate(queries)]
    if kind == "bank":
        outs, dqs = [], []
        total = torch.zeros(values.shape, device=values.device, dtype=torch.float64)
        for i, (query, upstream) in enumerate(zip(queries, grads)):
            out, dv, dq = _exact_read(values[: i + 1], query, upstream)
            outs.append(out)
            dqs.append(dq)
            total[: i + 1] += dv
        return {"out": outs, "dv": list(total.unbind(0)), "dq": dqs}
    out, dv, dq = _exact_read(values, queries[0], grads[0])
    return {"out": out, "dv": list(dv.unbind(0)) if kind == "list" else dv, "dq": dq}
