"""Host-side checks of the several-slot bank gather (no launch, no GPU)."""

from __future__ import annotations

from attnres import _native
from attnres.shared import _GatherRead

_FAKE = 0x7F0000001000


def _call(lib, reads, count, *, n_slots=4, base=None, dtype=0, partial=_FAKE, slot_stride=256, values=_FAKE, grad=_FAKE):
    return lib.attnres_hip_bank_gather_slots(values, 64, slot_stride, n_slots, 4, 64, reads, count, base, grad, dtype,
                                             partial, None)


def test_bank_gather_slots_checks_its_arguments():
    lib = _native.load()
    reads = (_GatherRead * 49)(*[(_FAKE, _FAKE, _FAKE, 9, 5, 16)] * 49)
    assert _call(lib, reads, 2, n_slots=2) == _native.ERR_SHAPE and b"n_slots" in lib.attnres_hip_last_error()
    assert _call(lib, reads, 49) == _native.ERR_SHAPE and b"at most 48 reads" in lib.attnres_hip_last_error()
    # the entry has no accumulate argument, and FP32 gradients take one launch too
    assert b"accumulate" not in lib.attnres_hip_last_error() and b"BF16" not in lib.attnres_hip_last_error()
    assert _call(lib, reads, 0) == _native.ERR_SHAPE
    assert _call(lib, reads, 2, partial=None) == _native.ERR_NULL_POINTER
    assert _call(lib, reads, 2, values=None) == _native.ERR_NULL_POINTER
    assert _call(lib, reads, 2, grad=None) == _native.ERR_NULL_POINTER
    assert _call(lib, reads, 2, dtype=2) == _native.ERR_SHAPE
    assert _call(lib, reads, 2, slot_stride=-1) == _native.ERR_STRIDE
    reads[1].position = 2  # slot 3 would be position -1
    assert _call(lib, reads, 2) == _native.ERR_SHAPE and b"position 2 outside 3..8" in lib.attnres_hip_last_error()
    reads[1].position, reads[1].rank = 5, 32
    assert _call(lib, reads, 2) == _native.ERR_SHAPE and b"one rank" in lib.attnres_hip_last_error()
