"""fmoe_permute and fmoe_permute_backward refuse bad arguments before any GPU work."""
from __future__ import annotations

import pytest

from fastmoe_amd import _abi

DEV = 0x10000  # never dereferenced: every call below is refused


def _permute(**over):
    a = dict(ids=DEV, id_dtype=_abi.I64, gates=DEV, gate_dtype=_abi.F32, T=4, k=2, E=8,
             row_bytes=32, x=DEV, stride=32, counts=DEV, offsets=DEV, rev=DEV, sorted=DEV,
             slot_pos=DEV, status=DEV, out=DEV, ws=DEV * 256)
    a.update(over)
    return _abi.lib().fmoe_permute(*a.values(), None)


@pytest.mark.parametrize("over,status", [
    ({"T": 0}, _abi.EINVAL), ({"k": 0}, _abi.EINVAL), ({"E": 0}, _abi.EINVAL),
    ({"E": 4097}, _abi.EINVAL), ({"id_dtype": _abi.F32}, _abi.EINVAL),
    ({"gate_dtype": _abi.I64}, _abi.EINVAL), ({"ids": None}, _abi.EINVAL),
    ({"out": None}, _abi.EINVAL), ({"x": None}, _abi.EINVAL), ({"status": None}, _abi.EINVAL),
    ({"row_bytes": 0}, _abi.EINVAL), ({"row_bytes": 31}, _abi.EINVAL),
    ({"stride": 16}, _abi.EINVAL), ({"row_bytes": 1 << 31, "stride": 1 << 31}, _abi.ERANGE),
    ({"T": 1 << 30, "k": 4}, _abi.ERANGE),
    ({"T": 4097, "ws": None}, _abi.EINVAL),          # past the one launch: needs its workspace
    ({"T": 4097, "ws": DEV * 256 + 8}, _abi.EINVAL),
])
def test_permute_refuses(over, status):
    assert _permute(**over) == status
    assert b"fmoe_permute" in _abi.lib().fmoe_last_error()


def _backward(**over):
    a = dict(slot_pos=DEV, T=4, k=2, D=16, dtype=_abi.BF16, rows=DEV, gx=DEV, gs=DEV,
             gate_dtype=_abi.F32, gg=DEV)
    a.update(over)
    return _abi.lib().fmoe_permute_backward(*a.values(), None)


@pytest.mark.parametrize("over,status", [
    ({"T": 0}, _abi.EINVAL), ({"k": 0}, _abi.EINVAL), ({"k": 65}, _abi.EINVAL),
    ({"D": 0}, _abi.EINVAL), ({"dtype": _abi.I32}, _abi.EINVAL), ({"rows": None}, _abi.EINVAL),
    ({"gx": None}, _abi.EINVAL), ({"slot_pos": None}, _abi.EINVAL), ({"gg": None}, _abi.EINVAL),
    ({"gs": None}, _abi.EINVAL), ({"gate_dtype": _abi.I64}, _abi.EINVAL),
    ({"T": 1 << 30}, _abi.ERANGE), ({"D": 1 << 29}, _abi.ERANGE),
])
def test_permute_backward_refuses(over, status):
    assert _backward(**over) == status
    assert b"fmoe_permute_backward" in _abi.lib().fmoe_last_error()


def test_small_limit():
    assert _abi.lib().fmoe_permute_small_max_slots() == 4096
