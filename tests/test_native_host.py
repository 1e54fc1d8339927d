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
    monkeypatch.setattr(native.WeightSteps, "_NO_PAIR", {0: tv.from_blob(0x7D0000000000, [32], tv.int32, 0)})
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


@pytest.fixture
def products(monkeypatch):
    """The argument blocks that reach cumm_hip_gemm and cumm_hip_gemm_in_workspace, in order; host memory
    stands for the workspaces."""
    from cumm_amd.gemm import main
    real, made = _capi.lib(), []

    class Library:
        def __getattr__(self, name):
            if name not in ("cumm_hip_gemm", "cumm_hip_gemm_in_workspace", "cumm_hip_stream_is_capturing"):
                return getattr(real, name)
            if name == "cumm_hip_stream_is_capturing":
                return lambda stream: 0

            def entry(desc, args, stream):
                made.append((name, _capi.GemmArgs.from_buffer_copy(args._obj), stream))
                return 0
            return entry
    monkeypatch.setattr(_capi, "_lib", Library())
    monkeypatch.setattr(main, "empty", lambda shape, dtype, device: tv.Tensor(shape, dtype))
    monkeypatch.setattr(main._Slots, "_device", staticmethod(lambda: 0))
    monkeypatch.setattr(main._Slots, "_spare", {})
    monkeypatch.setattr(native.WeightSteps, "_NO_PAIR", {0: tv.from_blob(0x7D0000000000, [32], tv.int32, 0)})
    return made


def _wide_operands(kv, counts, k_out=K, c_in=C):
    """Gradients and features that are columns of wider tensors: one product per offset."""
    blob = lambda at, shape, dtype: tv.from_blob(at, shape, dtype, 0)
    lists = SimpleNamespace(pair_in=blob(0x7F0000000000, [kv, 50000], tv.int32), pair_out=blob(0x7F1000000000, [kv, 50000], tv.int32),
                            counts=np.asarray(counts))
    return (blob(0x7F2000000000, [ROWS, k_out + 8], tv.float16).slice_axis(1, 0, k_out),
            blob(0x7F3000000000, [ROWS, c_in + 8], tv.float16).slice_axis(1, 0, c_in), blob(0x7F4000000000, [k_out, kv, c_in], tv.float16),
            lists)


def test_a_plan_of_single_products_runs_again_on_other_tensors(products):
    counts = [5000, 0, 12, 300, 40000]
    plan = native.plan_backward_weight(*_wide_operands(5, counts), stream=3)
    assert isinstance(plan, native.WeightSteps) and plan.launches == 5
    for early in (lambda: plan.rebind(1 << 20, 2 << 20, 3 << 20, 0), plan.release):
        with pytest.raises(RuntimeError, match="not run yet"):
            early()
    plan()
    first = products[:]
    assert [a.k for _, a, _ in first] == [5000, 32, 12, 300, 40000] and {s for _, _, s in first} == {3}
    # products with pairs enough share one workspace, the others have none
    spread = [name == "cumm_hip_gemm_in_workspace" for name, _, _ in first]
    assert spread == [True, False, False, True, True]
    assert len({a.workspace for (_, a, _), w in zip(first, spread) if w}) == 1
    assert all(a.workspace is None for (_, a, _), w in zip(first, spread) if not w)
    plan.release()
    assert plan.launches == 5
    with pytest.raises(RuntimeError, match="released"):
        plan()
    del products[:]
    base = 0x600000000000
    plan.rebind(base, base + (1 << 30), base + (2 << 30), 9)
    for (name, a, stream), (was_name, was, _) in zip(products, first):
        assert name == was_name and stream == 9 and (a.m, a.n, a.k) == (was.m, was.n, was.k)
        assert (a.ptr_A, a.ptr_B) == (base, base + (1 << 30))
        assert a.ptr_C == a.ptr_D == base + (2 << 30) + (was.ptr_C - 0x7F4000000000)
        assert (a.indiceA, a.indiceBorC) == (was.indiceA, was.indiceBorC)
    other = {a.workspace for (_, a, _), w in zip(products, spread) if w}
    assert len(other) == 1 and other != {a.workspace for (_, a, _), w in zip(first, spread) if w}      # (another stream)


def test_slices_are_what_the_caller_asks_for_where_no_workspace_spreads_the_pairs(products):
    """Outputs of more tiles than the spread kernel takes; with few pairs and one slice as it was."""
    workspace = tv.from_blob(0x7E0000000000, [1 << 20], tv.uint8, 0)
    operands = _wide_operands(3, [40000, 100, 16384], k_out=1088, c_in=1024)
    native.backward_weight(*operands, split_k_slices=4, workspace=workspace)
    assert [(a.split_k_slices, name) for name, a, _ in products] == [(4, "cumm_hip_gemm"), (1, "cumm_hip_gemm"), (4, "cumm_hip_gemm")]
    assert all(a.workspace == (0x7E0000000000 if a.split_k_slices > 1 else None) for _, a, _ in products)
    del products[:]
    native.backward_weight(*_wide_operands(2, [40000, 100]), split_k_slices=4)
    assert [(a.split_k_slices, name) for name, a, _ in products] == [(1, "cumm_hip_gemm_in_workspace"), (1, "cumm_hip_gemm")]


@pytest.fixture
def recording(products, monkeypatch):
    """``products``, and whether the streams are recorded: nothing may be allocated then."""
    from cumm_amd.gemm import main
    recorded, plain = [1], _capi.lib()

    class Library:
        def __getattr__(self, name):
            if name == "cumm_hip_stream_is_capturing":
                return lambda stream: recorded[0]
            if name == "cumm_hip_wgrad_pairs":
                return lambda *args: products.append((name, args[-3], args[-1])) or 0
            return getattr(plain, name)

    def empty(shape, dtype, device):
        assert not recorded[0]
        return tv.Tensor(shape, dtype)
    monkeypatch.setattr(_capi, "_lib", Library())
    monkeypatch.setattr(main, "empty", empty)
    return recorded


def test_a_recorded_run_has_no_workspace_but_the_callers(products, recording):
    """The graph may outlive the plan, whose workspace others get then."""
    counts = [5, 0, 96]
    operands = _operands(3, counts)
    dout, inp, dweight, lists = operands
    workspace = tv.from_blob(0x7E0000000000, [1 << 28], tv.uint8, 0)

    def single_products(at, stream):
        assert [(name, a.k) for name, a, _ in products] == [("cumm_hip_gemm", k) for k in (5, 32, 96)]
        for r, (_, a, s) in enumerate(products):
            assert (a.ptr_A, a.ptr_B, a.ptr_C, a.workspace, s) == (at[0], at[1], at[2] + r * C * 2, None, stream)
        assert products[2][1].indiceA == lists.pair_out.byte_pointer() + 2 * MOST * 4
        del products[:]
    here = [t.byte_pointer() for t in (dout, inp, dweight)]
    native.backward_weight(*operands, stream=4)
    single_products(here, 4)
    native.backward_weight(*operands, stream=4, workspace=workspace)
    assert products == [("cumm_hip_wgrad_pairs", 0x7E0000000000, 4)]
    del products[:]
    plan = native.plan_backward_weight(*operands, stream=4)
    for recorded in (0, 1, 0):
        recording[0] = recorded
        for run, at, stream in ((plan, here, 4), (lambda: plan.rebind(1 << 40, 2 << 40, 3 << 40, 5), [i << 40 for i in (1, 2, 3)], 5)):
            run()
            if recorded:
                single_products(at, stream)
            else:
                assert [(name, s) for name, _, s in products] == [("cumm_hip_wgrad_pairs", stream)]
                del products[:]


def test_a_plan_of_single_products_that_was_recorded_first(products, recording):
    counts = [5000, 0, 300]
    plan = native.plan_backward_weight(*_wide_operands(3, counts), stream=3)
    plan()
    assert [(name, a.workspace) for name, a, _ in products] == [("cumm_hip_gemm", None)] * 3
    first = products[:]
    plan.release()
    assert plan.launches == 3
    base = 0x600000000000
    for recorded in (1, 0, 0):
        recording[0] = recorded
        del products[:]
        plan.rebind(base, base + (1 << 30), base + (2 << 30), 9)
        want = ["cumm_hip_gemm_in_workspace" if k > 32 and not recorded else "cumm_hip_gemm" for k in (5000, 32, 300)]
        assert [name for name, _, _ in products] == want
        for (name, a, stream), (_, was, _) in zip(products, first):
            assert (a.ptr_A, a.ptr_B, stream, a.k) == (base, base + (1 << 30), 9, was.k) and bool(a.workspace) == ("in_work" in name)
            assert a.ptr_C == base + (2 << 30) + (was.ptr_C - 0x7F4000000000) and a.stride_A == was.stride_A == K + 8
    # on a stream of its own, recorded: nothing is allocated for it, and the entry point uses no workspace
    recording[0] = 1
    plan.rebind(base, base + (1 << 30), base + (2 << 30), 10)


def test_lists_of_2_to_the_29_pairs_and_more_are_refused():
    """Their bytes do not fit the 31 bits of an offset inside a list."""
    lib = _capi.lib()
    for counts, taken in (([(1 << 29) - 1], True), ([1 << 29], False), ([5, 1 << 30, 7], False), ([2147483647], False), ([-1], False)):
        c = np.array(counts, np.int32)
        need = lib.cumm_hip_wgrad_pairs_workspace(c.ctypes.data, len(counts), 64, 64)
        assert (need > 0) == taken and (taken or need == -1), counts
        if not taken:
            at = 1 << 20      # (never read: the counts are refused first)
            assert lib.cumm_hip_wgrad_pairs(at, at, at, at, at, c.ctypes.data, len(counts), 1 << 31, 10, 10, 64, 64, tv.float16, at,
                                            1 << 40, None) == _capi.EINVAL


def test_what_one_call_does_not_take_goes_out_as_single_products(products):
    """4096 blocks of 64 x 64 channels and more; the plan takes a block less in one call."""
    for k_out, c_in, single in ((4096, 4096, True), (4096, 4032, False)):
        blob = lambda at, shape, dtype: tv.from_blob(at << 32, shape, dtype, 0)
        lists = SimpleNamespace(pair_in=blob(0x7F00, [2, 100], tv.int32), pair_out=blob(0x7F01, [2, 100], tv.int32),
                                counts=np.array([100, 7]))
        operands = (blob(0x7F02, [ROWS, k_out], tv.float16), blob(0x7F03, [ROWS, c_in], tv.float16),
                    blob(0x7F04, [k_out, 2, c_in], tv.float16), lists)
        assert isinstance(native.plan_backward_weight(*operands), native.WeightSteps) == single
        if single:
            native.backward_weight(*operands)
            assert [(name, a.k) for name, a, _ in products] == [("cumm_hip_gemm", 100), ("cumm_hip_gemm", 7)]
