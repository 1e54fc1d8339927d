"""Checks of the per-offset weight gradient that need no GPU (cumm_amd/conv/native.py): the library's entry
point is replaced by one that keeps its arguments, addresses are never dereferenced."""
import ctypes
from types import SimpleNamespace

import numpy as np
import pytest

from cumm_amd import _capi
from cumm_amd import tensorview as tv
from cumm_amd.conv import native

ROWS, K, C, MOST = 500, 24, 40, 96


@pytest.fixture
def calls(monkeypatch):
    real, made = _capi.lib(), []

    class Library:
        def __getattr__(self, name):
            if name != "cumm_hip_wgrad_pairs":
                return getattr(real, name)

            def entry(dw, dout, inp, pair_out, pair_in, counts, lists, stride, *rest):
                made.append((np.ctypeslib.as_array(ctypes.cast(counts, ctypes.POINTER(ctypes.c_int32)), (lists,)).copy(), stride))
                return 0
            return entry
    monkeypatch.setattr(_capi, "_lib", Library())
    return made


def _operands(kv, counts, device=0, list_device=0, list_dtype=tv.int32):
    at = iter(range(0x7F0000000000, 0x7FF000000000, 1 << 32))

    def blob(shape, dtype, where):
        if where < 0:
            return tv.zeros(shape, dtype)
        return tv.from_blob(next(at), shape, dtype, where)
    lists = SimpleNamespace(pair_in=blob([kv, MOST], list_dtype, list_device), pair_out=blob([kv, MOST], list_dtype, list_device),
                            counts=np.asarray(counts))
    return (blob([ROWS, K], tv.float16, device), blob([ROWS, C], tv.float16, device), blob([K, kv, C], tv.float16, device), lists)


def _run(operands):
    native.backward_weight(*operands, workspace=tv.from_blob(0x7E0000000000, [1 << 28], tv.uint8, 0))


def test_host_tensors_other_devices_and_other_list_types_are_refused(calls):
    _run(_operands(3, [5, 0, 96]))
    assert len(calls) == 1
    with pytest.raises(RuntimeError, match="device tensors"):
        _run(_operands(3, [5, 0, 96], device=-1, list_device=-1))
    for devices in ((-1, 0), (0, -1), (0, 1), (1, 0)):
        with pytest.raises(ValueError, match="same device"):
            _run(_operands(3, [5, 0, 96], *devices))
    with pytest.raises(RuntimeError, match="dtype"):
        _run(_operands(3, [5, 0, 96], list_dtype=tv.int64))
    assert len(calls) == 1


@pytest.mark.parametrize("counts", [[97], [5000], [-3], [96, 1000, -1, 0, 12]])
def test_a_count_ends_with_its_list(calls, counts):
    _run(_operands(len(counts), counts))
    assert calls[0][0].tolist() == [min(max(c, 0), MOST) for c in counts] and calls[0][1] == MOST
