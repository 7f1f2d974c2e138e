"""Several reads of shared sources, with the source gradients summed inside
the backward kernels: ``SharedSources`` (a fixed list read by several
queries) and ``SourceBank`` (sources appended one at a time and read as
prefixes, the residual stream of a Full-schedule model).

Autograd sums the gradients of a tensor used by several reads with separate
add kernels after each read's backward: for a source of N x D BF16 elements
every further read costs a pass that reads two gradient buffers and writes a
third.  ``SharedSources`` instead gives every read of the same sources one set
of gradient buffers: the first backward writes them, each later backward
adds its dv in the kernel (``attnres_hip_sources_backward_accumulate``: one
extra read of the buffer, no add kernel), and the sources receive the sums
once every read's backward has run.

    bank = SharedSources(sources)             # ordered list of BF16 [..., D] tensors
    out_a = bank.read(query_a)                # same result as attnres(sources, query_a)
    out_b = bank.read(query_b, scale=0.5)
    loss(out_a, out_b).backward()             # sources get d/d(source) summed over both reads

The ordering uses a token: the reads take a zero-size tensor produced from
the sources by one autograd node, so autograd runs that node's backward --
which hands the summed buffers to the sources -- only after every read that
received a gradient.  Each backward pass (autograd graph task) starts a
fresh sum, also after a pass that stopped short of the sources (e.g.
``torch.autograd.grad`` with respect to the queries only).  Eager mode only
(the bank holds state between the reads' backward calls); first-order
gradients, like the read itself.

The autograd nodes hold the buffers and the per-pass bookkeeping in a state
object that holds no token, so the buffers are freed with the graph, without
waiting for Python's cycle collector (a node that held the bank itself would
close a cycle bank -> token -> node -> bank).  A ``SourceBank``'s nodes and
state are C++ (`csrc/attnres_autograd.cpp`): the backward of a read or a push
runs without Python.

The reference has no counterpart: its shared sources' gradients are summed
by autograd (the Block-schedule reads of `benchmarks/model.py:306-338`).
"""

from __future__ import annotations

import ctypes
from typing import Sequence

import torch
from torch import Tensor

from . import _native
from ._ops import _contiguous, _dq_workspace, _on_device, _source_table, _stream, sources_forward_impl
from ._sources import _EPS, _MAX_SOURCES, _MAX_WIDTH, check_query, check_sources

_MAX_GATHER_READS = 48  # attnres_hip.h ATTNRES_MAX_GATHER_READS
# A BF16 source's gathered gradient is stored as BF16 by the gather itself
# when one launch covers its reads (else FP32, converted afterwards).
_BF16_GATHER = True


class _GatherRead(ctypes.Structure):
    """attnres_hip.h ``attnres_gather_read``."""

    _fields_ = [("grad_out", ctypes.c_void_p), ("query_row", ctypes.c_void_p), ("coef", ctypes.c_void_p),
                ("n_sources", ctypes.c_int64), ("position", ctypes.c_int64), ("rank", ctypes.c_int64)]


_GRAPH_TASK_ID = getattr(torch._C, "_current_graph_task_id", None)


def _pass_id() -> int:
    """The running backward pass: autograd's graph-task id (-1 outside one).
    No public torch API tells one backward pass from the next; a torch build
    without this query cannot run shared-source reads and says so."""
    if _GRAPH_TASK_ID is None:
        raise RuntimeError("SharedSources and SourceBank need torch._C._current_graph_task_id, "
                           "which this torch build does not provide")
    return _GRAPH_TASK_ID()


class _SharedState:
    """The sources and this pass's gradient sums, used by the nodes of a
    ``SharedSources``."""

    def __init__(self, sources: tuple[Tensor, ...]) -> None:
        self.sources = sources
        self._grads: list[Tensor] | None = None
        self._pass = -1

    def _backward(self, query: Tensor, out: Tensor, out_refine: Tensor, grad_out: Tensor,
                  logit: Tensor, inv_rms: Tensor, stats: Tensor, scale: float) -> Tensor:
        """One read's backward: dv into the shared buffers (written by the
        first read of this pass, accumulated by the others); returns dq."""
        lib = _native.load()
        first = self.sources[0]
        count, width = len(self.sources), int(first.shape[-1])
        tokens = out.numel() // width
        rank = query.numel()
        device = first.device
        current = _pass_id()
        accumulate = self._grads is not None and self._pass == current
        if not accumulate:  # first read of this pass (an earlier pass may have left its sums untaken)
            self._grads = [torch.empty(first.shape, device=device, dtype=torch.bfloat16) for _ in range(count)]
            self._pass = current
        flags = (ctypes.c_uint8 * count)(*([1 if accumulate else 0] * count))
        grad_pointers = (ctypes.c_void_p * count)(*[grad.data_ptr() for grad in self._grads])
        prepared, pointers, row_strides = _source_table(list(self.sources))
        grad_query = torch.empty((rank,), device=device, dtype=torch.bfloat16)
        workspace = _dq_workspace(lib, tokens, width, rank, device)
        grad_out = _contiguous(grad_out.to(torch.bfloat16))
        with _on_device(device):
            status = lib.attnres_hip_sources_backward_accumulate(
                pointers, row_strides, count, tokens, width, query.data_ptr(), rank, scale,
                _contiguous(out).data_ptr(), _contiguous(out_refine).data_ptr(), grad_out.data_ptr(),
                _contiguous(logit).data_ptr(), _contiguous(inv_rms).data_ptr(), _contiguous(stats).data_ptr(),
                grad_pointers, grad_query.data_ptr(), workspace.data_ptr(), workspace.numel(), flags,
                _stream(device))
        del prepared
        _native.check(status, "attnres shared-source backward")
        return grad_query

    def _take_grads(self) -> list[Tensor] | None:
        grads, self._grads = self._grads, None
        return grads if self._pass == _pass_id() else None


class SharedSources:
    """An ordered list of BF16 sources read by several queries (see module doc)."""

    def __init__(self, sources: Sequence[Tensor]) -> None:
        if not isinstance(sources, (list, tuple)) or not sources:
            raise TypeError("sources must be a non-empty list or tuple of tensors")
        first = sources[0]
        if not isinstance(first, Tensor):
            raise TypeError("values must contain only tensors")
        probe = torch.empty(1, device=first.device, dtype=torch.bfloat16)
        checked, _, _ = check_sources(tuple(sources), probe, _EPS, 1.0)
        if not checked[0].is_cuda:
            raise RuntimeError("attnres requires CUDA (ROCm/HIP) device tensors")
        self._state = _SharedState(checked)
        self._token = _Gather.apply(self._state, *checked)

    @property
    def sources(self) -> tuple[Tensor, ...]:
        return self._state.sources

    def __len__(self) -> int:
        return len(self.sources)

    def read(self, query: Tensor, *, eps: float = _EPS, scale: float = 1.0) -> Tensor:
        """``attnres(sources, query, eps=eps, scale=scale)`` with the source
        gradients summed in the kernels across this bank's reads."""
        _, eps_value, scale_value = check_sources(self.sources, query, eps, scale)
        if not _needs_gradients(query, self._token):  # the forward alone: nothing saved
            return sources_forward_impl(list(self.sources), _contiguous(query), eps_value, scale_value, False,
                                        pooled=True)[0]
        return _Read.apply(self._state, self._token, query, eps_value, scale_value)


class _Gather(torch.autograd.Function):
    """The bank's autograd node: its backward hands the summed gradients to
    the sources after every read's backward."""

    @staticmethod
    def forward(ctx, bank: _SharedState, *sources: Tensor) -> Tensor:
        ctx.bank = bank
        return sources[0].new_empty((0,))

    @staticmethod
    def backward(ctx, _token_grad):
        grads = ctx.bank._take_grads()
        count = len(ctx.bank.sources)
        if grads is None:
            return (None,) * (count + 1)
        return (None, *[g if need else None for g, need in zip(grads, ctx.needs_input_grad[1:])])


class _Read(torch.autograd.Function):
    @staticmethod
    def forward(ctx, bank: _SharedState, token: Tensor, query: Tensor, eps: float, scale: float) -> Tensor:
        query = _contiguous(query)
        # always saved: the accumulating kernels read the refinement
        out, out_refine, logit, inv_rms, stats = sources_forward_impl(list(bank.sources), query, eps, scale, True,
                                                                      pooled=True)
        ctx.bank = bank
        ctx.scale = scale
        ctx.token_device = token.device
        ctx.save_for_backward(query, out, out_refine, logit, inv_rms, stats)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        query, out, out_refine, logit, inv_rms, stats = ctx.saved_tensors
        grad_query = ctx.bank._backward(query, out, out_refine, grad_out, logit, inv_rms, stats, ctx.scale)
        token_grad = torch.empty((0,), device=ctx.token_device)
        return None, token_grad, grad_query if ctx.needs_input_grad[2] else None, None, None


class SourceBank:
    """Sources kept in numbered slots of one packed BF16 buffer and read as
    slot lists: the residual stream of a Full- or Block-schedule model.

    Full schedule (read i sees every source pushed before it)::

        bank = SourceBank(capacity=2 * layers + 1)
        bank.push(embedding)                      # slot 0; any float dtype, shape [..., D]
        x = bank.read(query_0)                    # attnres over slot 0 (BF16 out)
        bank.push(sublayer(x.to(dtype)))          # slot 1
        x = bank.read(query_1)                    # over slots 0..1, ...

    Block schedule (a read sees the completed blocks, slots 0..k-1, plus the
    running partial sum of the current block in some other slot)::

        bank.push(embedding, slot=0)
        bank.push(first_emitted, slot=p)          # the partial starts as one output
        x = bank.read(query, count=1, tail=p)     # attnres(embedding, partial)
        partial = bank.push_sum(partial, emitted, slot=q)   # partial + emitted, one pass

    Each source is converted to BF16 once, into its slot, so a read passes
    slot rows (the prefix view ``buffer[:count]``, or a list of slot pointers
    when a tail slot is added) with no per-read conversion or stack.
    ``push_sum`` adds the block's partial and the new output and writes the
    sum (in their dtype, returned) and its BF16 copy (into the slot) in one
    kernel (``attnres_hip_partial_sum``).

    Gradients (``gradients="gather"``, the default): a read's backward writes
    no dv rows, only its dq and the per-token coefficients of its dv
    (``attnres_hip_{packed,sources}_backward_coef``), and keeps its BF16 dO.
    Slot i's gradient is formed once, when the slot's push node runs its
    backward, by ``attnres_hip_bank_gather_slots``: one FP32 pass over the dO
    rows of the reads that saw slot i.  From nine such reads on the same pass
    also forms the sums of the three slots before it, where the backward pass
    computes their gradients too, and these add their later reads to them (12
    more bytes per element of a source at the peak of the pass).  The ordering
    uses one chain of zero-size tokens: every push node takes the token of the
    push before it, and a read takes the latest token, so a push node's backward
    runs after that of every read made after the push (those that saw the slot
    among them), and a read has one token input however many slots it reads.
    ``gradients="accumulate"`` instead adds every read's FP32 dv into one FP32
    ``[capacity, ..., D]`` buffer in the backward kernel
    (``attnres_hip_{packed,sources}_backward_accumulate_f32``:
    a read-modify-write of the sum per read).  Either way the sums are FP32
    without BF16 rounding of the per-read dv, and reach the source in its
    dtype.  Eager mode only; one bank per forward pass.
    """

    def __init__(self, capacity: int, *, gradients: str = "gather") -> None:
        if isinstance(capacity, bool) or not isinstance(capacity, int) or not 1 <= capacity <= _MAX_SOURCES:
            raise ValueError(f"capacity must be an integer in 1..{_MAX_SOURCES}")
        if gradients not in ("gather", "accumulate"):
            raise ValueError("gradients must be 'gather' or 'accumulate'")
        self.capacity = capacity
        self.gradients = gradients
        self._state = None  # the C++ nodes' slots (`BankState`), allocated by the first push
        self._nodes = None
        self._shape: torch.Size | None = None
        self._device: torch.device | None = None
        self._pushed: list[bool] = [False] * capacity
        self._token: Tensor | None = None  # the latest push's token

    def __len__(self) -> int:
        """Number of pushed slots."""
        return sum(self._pushed)

    def _claim(self, source: Tensor, slot: int | None) -> int:
        if not isinstance(source, Tensor) or not source.is_floating_point():
            raise TypeError("a source must be a floating-point tensor")
        if not source.is_cuda:
            raise RuntimeError("attnres requires CUDA (ROCm/HIP) device tensors")
        if slot is None:
            free = [i for i, pushed in enumerate(self._pushed) if not pushed]
            if not free:
                raise ValueError("the source bank is full")
            slot = free[0]
        if isinstance(slot, bool) or not isinstance(slot, int) or not 0 <= slot < self.capacity:
            raise ValueError(f"slot must be an integer in 0..{self.capacity - 1}")
        if self._pushed[slot]:
            raise ValueError(f"slot {slot} already holds a source")
        if self._state is None:
            if source.ndim < 1 or source.numel() == 0 or not 1 <= source.shape[-1] <= _MAX_WIDTH:
                raise ValueError("each source must have shape [...,D]")
            self._nodes = _native.load_autograd()
            self._state = self._nodes.BankState(self.capacity, self.gradients == "gather", _BF16_GATHER, source)
            self._shape, self._device = source.shape, source.device
        elif source.shape != self._shape or source.device != self._device:
            raise ValueError("all source tensors must have the same logical shape and device")
        return slot

    def push(self, source: Tensor, *, slot: int | None = None) -> int:
        """Store ``source`` (``[..., D]``, any float dtype, on the GPU) in
        ``slot`` (default: the lowest free one); returns the slot."""
        slot = self._claim(source, slot)
        self._token = self._nodes.bank_push(self._state, slot, source, self._token)
        self._pushed[slot] = True
        return slot

    def push_sum(self, prev: Tensor, emitted: Tensor, *, slot: int | None = None) -> Tensor:
        """``prev + emitted`` (FP32 or BF16, same shape and dtype), returned in
        that dtype and stored as BF16 in ``slot`` -- one kernel for the
        Block schedule's partial sum and its BF16 copy."""
        if not isinstance(prev, Tensor) or not isinstance(emitted, Tensor):
            raise TypeError("push_sum takes two tensors")
        if prev.shape != emitted.shape or prev.dtype != emitted.dtype or prev.device != emitted.device:
            raise ValueError("push_sum needs tensors of one shape, dtype and device")
        if prev.dtype not in (torch.float32, torch.bfloat16):
            raise TypeError("push_sum supports float32 and bfloat16 tensors")
        slot = self._claim(emitted, slot)
        partial, self._token = self._nodes.bank_push_sum(self._state, slot, prev, emitted, self._token)
        self._pushed[slot] = True
        return partial

    def read(self, query: Tensor, *, count: int | None = None, tail: int | None = None, eps: float = _EPS,
             scale: float = 1.0) -> Tensor:
        """``attnres`` over slots ``0..count-1`` (default: every pushed slot,
        which must then be ``0..len-1``) followed by slot ``tail`` if given; BF16."""
        if count is None:
            if tail is not None:
                raise ValueError("a read with a tail slot needs count")
            count = len(self)
        if isinstance(count, bool) or not isinstance(count, int) or not 0 <= count <= self.capacity:
            raise ValueError("count must be a number of leading slots")
        if not all(self._pushed[:count]):
            raise ValueError("count must select pushed slots 0..count-1")
        if tail is not None:
            if isinstance(tail, bool) or not isinstance(tail, int) or not count <= tail < self.capacity \
                    or not self._pushed[tail]:
                raise ValueError("tail must be a pushed slot after the leading ones")
        elif count == 0:
            raise ValueError("a read needs at least one source")
        # the slots were checked at their push: BF16 rows [..., D] on one device
        eps_value, scale_value = check_query(query, self._shape[-1], self._device, eps, scale)
        return self._nodes.bank_read(self._state, count, -1 if tail is None else tail, query, eps_value, scale_value,
                                     self._token)


def _needs_gradients(query: Tensor, token: Tensor | None) -> bool:
    """Whether autograd will want this read's gradients: grad mode on and the
    query or the sources (through the container's token) requiring grad.
    Otherwise a read runs the forward alone, with no refinement bytes or
    saved state, and the same output bits."""
    return torch.is_grad_enabled() and (query.requires_grad or (token is not None and token.requires_grad))


__all__ = ["SharedSources", "SourceBank"]
