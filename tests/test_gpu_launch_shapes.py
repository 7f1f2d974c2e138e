"""The kernel a read takes depends on how many tokens it has (one workgroup
per token, one token per group, blocks of two or four tokens, rows in flight);
a token's output, saved statistics and value gradient do not.  Every geometry
is read with token counts on both sides of each rule, aligned and not, and
must give the same bits for the same tokens."""

from __future__ import annotations

import math

import pytest
import torch

from attnres import _native, _ops

pytestmark = pytest.mark.gpu


def _backward(values, query, state, grad, save):
    sources, tokens, width = values.shape
    lib = _native.load()
    out, refine, logit, inv_rms, stats = state
    dv = torch.empty(sources, tokens, width, device="cuda", dtype=torch.bfloat16)
    dq = torch.empty(query.numel(), device="cuda", dtype=torch.bfloat16)
    workspace = torch.empty(lib.attnres_hip_dq_workspace_elems(tokens, width, query.numel()), device="cuda")
    status = lib.attnres_hip_packed_backward(
        values.data_ptr(), values.stride(0), values.stride(1), sources, tokens, width, query.data_ptr(), query.numel(),
        1.0, out.data_ptr() if save else None, refine.data_ptr() if save else None, grad.data_ptr(), logit.data_ptr(),
        inv_rms.data_ptr(), stats.data_ptr(), dv.data_ptr(), dq.data_ptr(), workspace.data_ptr(), workspace.numel(),
        torch.cuda.current_stream().cuda_stream)
    _native.check(status, "packed backward")
    return dv


@pytest.mark.parametrize("sources", [2, 6, 14, 25])
@pytest.mark.parametrize("width,rank,offset", [
    (256, 256, 0), (200, 50, 0), (257, 257, 0), (512, 512, 0), (513, 128, 0), (640, 640, 0), (768, 768, 0), (768, 192, 1),
    (769, 769, 0), (896, 896, 0), (1024, 1024, 0), (1024, 256, 0), (1025, 1025, 0), (1280, 320, 0), (1536, 1536, 0),
    (1537, 385, 0), (1800, 1800, 0), (2048, 2048, 0), (2048, 700, 0), (2049, 2049, 0), (2560, 2560, 0), (2560, 640, 1),
    (2561, 2561, 0), (3072, 3072, 0), (3073, 768, 0), (4096, 4096, 0), (4096, 512, 0), (4097, 4097, 0), (5120, 1280, 0),
    (6144, 6144, 0), (6145, 1536, 0), (8192, 8192, 0),
])
def test_bits_do_not_depend_on_the_token_count(sources, width, rank, offset):
    largest = 17001 if width <= 1024 else 9001 if width <= 3072 else 4501
    largest = min(largest, 500_000_000 // (sources * width))
    print(f"launch shapes S={sources} D={width} R={rank} offset={offset} N<={largest}", flush=True)
    torch.manual_seed(width + sources)
    values = torch.randn(sources, largest, width + offset, device="cuda", dtype=torch.bfloat16)[..., offset:]
    query = (torch.randn(rank, device="cuda") * 3 / math.sqrt(rank)).to(torch.bfloat16)
    grad = torch.randn(largest, width, device="cuda", dtype=torch.bfloat16)
    save = _ops.saves_refinement(sources, width, rank)
    whole = _ops.packed_forward_impl(values, query, 2**-23, 1.0, save)
    whole_dv = _backward(values, query, whole, grad, save)
    for tokens in (37, 1000, 2600, 4095):
        if tokens >= largest:
            continue
        rows = values[:, :tokens]
        part = _ops.packed_forward_impl(rows, query, 2**-23, 1.0, save)
        dv = _backward(rows, query, part, grad[:tokens], save)
        torch.cuda.synchronize()
        assert torch.equal(part[0], whole[0][:tokens]), f"out of {tokens} tokens"
        assert not save or torch.equal(part[1], whole[1][:tokens]), f"refinement of {tokens} tokens"
        assert torch.equal(part[2], whole[2][:tokens]) and torch.equal(part[3], whole[3][:tokens])
        assert torch.equal(part[4], whole[4][:, :tokens]), f"stats of {tokens} tokens"
        assert torch.equal(dv, whole_dv[:, :tokens]), f"dv of {tokens} tokens"
