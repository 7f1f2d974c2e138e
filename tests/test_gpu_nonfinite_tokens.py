"""A token that holds NaN or infinite values changes no other token.

A group of the one-token forward streams the rows of one token after another
through the same registers, so the read has far more tokens than the groups a
persistent grid keeps resident: every group that meets a spoiled token also
forms clean ones after it.  For every row geometry and every number of sources
that may take that grid, the outputs, saved state and value gradients of the
clean tokens are the same bits with and without the spoiled ones.
"""

from __future__ import annotations

import math

import pytest
import torch

from attnres import _native, _ops

pytestmark = pytest.mark.gpu

_SOURCES = 13  # one past the reads that take a persistent grid


def _backward(rows, query, state, grad, save):
    sources, tokens, width = rows.shape
    lib = _native.load()
    out, refine, logit, inv_rms, stats = state
    dv = torch.empty(sources, tokens, width, device="cuda", dtype=torch.bfloat16)
    dq = torch.empty(query.numel(), device="cuda", dtype=torch.bfloat16)
    workspace = torch.empty(lib.attnres_hip_dq_workspace_elems(tokens, width, query.numel()), device="cuda")
    status = lib.attnres_hip_packed_backward(
        rows.data_ptr(), rows.stride(0), rows.stride(1), sources, tokens, width, query.data_ptr(), query.numel(), 1.0,
        out.data_ptr() if save else None, refine.data_ptr() if save else None, grad.data_ptr(), logit.data_ptr(),
        inv_rms.data_ptr(), stats.data_ptr(), dv.data_ptr(), dq.data_ptr(), workspace.data_ptr(), workspace.numel(),
        torch.cuda.current_stream().cuda_stream)
    _native.check(status, "packed backward")
    return dv


@pytest.mark.parametrize("layout", ["packed", "list"])
@pytest.mark.parametrize("width,rank", [
    (64, 64), (128, 40), (256, 256), (512, 512), (768, 768), (1000, 1000), (1024, 1024), (1025, 300), (1536, 1536),
    (2048, 2048), (2048, 512), (2560, 640), (3072, 3072), (4096, 4096), (4096, 1024), (4097, 4097), (5120, 1280),
    (6144, 6144), (8192, 8192),
])
def test_a_nonfinite_token_changes_no_other_token(width, rank, layout):
    # groups of a full grid: at most 8 workgroups per CU of 256 CUs, 256 lanes each
    lanes = 16 if width <= 128 else 32 if width <= 1024 else 64 if width <= 4096 else 256
    tokens = max(2 * 256 * (2048 // lanes) + 5, 3001) if lanes < 64 else 9001 if lanes == 64 else 3001
    print(f"non-finite tokens D={width} R={rank} N={tokens} {layout}", flush=True)
    torch.manual_seed(width + rank)
    values = torch.randn(_SOURCES, tokens, width, device="cuda", dtype=torch.bfloat16)
    query = (torch.randn(rank, device="cuda") / math.sqrt(rank)).to(torch.bfloat16)
    grad = torch.randn(tokens, width, device="cuda", dtype=torch.bfloat16)
    spoiled = {0: float("nan"), 7: float("inf"), 64: float("-inf"), 300: float("nan"), 1001: float("inf")}
    clean = torch.ones(tokens, device="cuda", dtype=torch.bool)
    clean[list(spoiled)] = False

    for sources in range(1, _SOURCES + 1):
        save = _ops.saves_refinement(sources, width, rank)

        def read():
            rows = values[:sources]
            if layout == "packed":
                state = _ops.packed_forward_impl(rows, query, 2**-23, 1.0, save)
            else:
                state = _ops.sources_forward_impl(list(rows.unbind(0)), query, 2**-23, 1.0, save)
            return (*state, _backward(rows, query, state, grad, save) if layout == "packed" else None)

        expected = read()
        kept = {}
        for n, value in spoiled.items():
            s, d = n % sources, (n * 37) % width
            kept[n] = (s, d, values[s, n, d].clone())
            values[s, n, d] = value
        actual = read()
        for n, (s, d, value) in kept.items():
            values[s, n, d] = value
        torch.cuda.synchronize()
        case = f"S={sources} D={width} R={rank}"
        assert torch.isfinite(expected[0]).all(), case
        for name, a, b in zip(("out", "refine", "logit", "inv_rms"), actual, expected):
            if name != "refine" or save:
                assert torch.equal(a[clean], b[clean]), f"{name} of {case}"
        assert torch.equal(actual[4][:, clean], expected[4][:, clean]), f"stats of {case}"
        if layout == "packed":
            assert torch.equal(actual[5][:, clean], expected[5][:, clean]), f"dv of {case}"
