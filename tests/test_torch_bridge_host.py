"""Host logic of the torch bridge that needs no GPU: the argument blocks of validated calls, whose addresses
are never dereferenced here."""
import os
import subprocess
import threading

import pytest

from cumm_amd import _capi
from cumm_amd import tensorview as tv
from cumm_amd.conv.main import ConvMainUnitTest
from cumm_amd.tensorview.gemm import ConvOpType, ConvParams

torch = pytest.importorskip("torch")


class _Recorder:
    """The library with some entry points replaced by what keeps their arguments."""

    def __init__(self, *names):
        self._real, self._names, self.calls = _capi.lib(), names, []

    def __getattr__(self, name):
        if name not in self._names:
            return getattr(self._real, name)

        def entry(*args):
            self.calls.append((name,) + tuple(type(a._obj).from_buffer_copy(a._obj) if hasattr(a, "_obj") else a for a in args))
            return 0
        return entry


@pytest.fixture
def recorded(monkeypatch):
    def use(*names):
        r = _Recorder(*names)
        monkeypatch.setattr(_capi, "_lib", r)
        return r
    return use


class _At:
    """What a call sees of a tensor: its address."""

    def __init__(self, address):
        self.address = address

    def data_ptr(self):
        return self.address

    def numel(self):
        return 1


N, C, KV = 1000, 64, 27


def _params(op, addresses, bias=None):
    at = lambda role, shape: tv.from_blob(addresses[role], shape, tv.float16, 0)
    blob = lambda shape, dtype: tv.from_blob(0x7E0000000000, shape, dtype, 0)
    p = ConvParams(3, op)
    p.conv_algo_desp = [d for d in ConvMainUnitTest.get_all_conv_algo_desp()
                        if d.dtype_a == tv.float16 and d.dtype_c == tv.float16 and ConvOpType(d.op_type) == op][0].copy()
    p.input, p.weight, p.output = at("input", [N, C]), at("weight", [C, KV, C]), at("output", [N, C])
    p.indices, p.mask_argsort = blob([KV, N], tv.int32), blob([N], tv.int32)
    p.mask = blob([N], tv.uint32)
    if op == ConvOpType.BackwardWeight:
        p.mask_width = 64
    if bias is not None:
        p.bias, p.beta = tv.from_blob(bias, [C], tv.float16, 0), 1.0
    return p


@pytest.mark.parametrize("op,with_bias", [(ConvOpType.Forward, False), (ConvOpType.Forward, True), (ConvOpType.BackwardInput, False),
                                          (ConvOpType.BackwardWeight, False)])
@pytest.mark.parametrize("shared", [(), ("input", "output"), ("input", "weight"), ("weight", "output"), ("input", "weight", "output")])
def test_a_call_keeps_its_tensors_apart_whatever_the_first_one_shared(recorded, op, with_bias, shared):
    """A block that was validated with tensors at one address, replayed with tensors at three."""
    from cumm_amd import torch_bridge as tb
    lib = recorded("cumm_hip_sparse_conv")
    first = {"input": 0x7F0000000000, "weight": 0x7F1000000000, "output": 0x7F2000000000}
    first.update({role: 0x7F3000000000 for role in shared})
    p = _params(op, first, bias=0x7F4000000000 if with_bias else None)
    ConvMainUnitTest.implicit_gemm2(p)
    roles = {role: _At(a) for role, a in first.items()}
    if with_bias:
        roles["bias"] = _At(0x7F4000000000)
    launch = tb._Launch.of(p, roles)
    new = {role: 0x600000000000 + (i << 32) for i, role in enumerate(roles)}
    launch(0, **{role: _At(a) for role, a in new.items()})
    args = lib.calls[-1][2]
    a, b, c = {ConvOpType.Forward: ("input", "weight", "output"), ConvOpType.BackwardInput: ("output", "weight", "input"),
               ConvOpType.BackwardWeight: ("output", "input", "weight")}[op]
    assert (args.ptr_A, args.ptr_B, args.ptr_C) == (new[a], new[b], new[c])
    assert args.ptr_D == new["bias" if with_bias else c]
    assert args.bias_pointer == (new["bias"] if with_bias else None)


def _geometry(monkeypatch, tb, n=1000, stream=1):
    """A submanifold geometry of ``n`` voxels as its constructor leaves it on ``stream``, in host memory; the
    second result lists what is recorded for another stream, by the address of its memory."""
    now, recorded = [stream], []
    monkeypatch.setattr(tb, "current_stream", lambda: now[0])
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: now[0])
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda t, s: recorded.append((t.untyped_storage().data_ptr(), s)))
    g = object.__new__(tb.SparseConvGeometry)
    g._stream, g._device, g.subm, g.kv, g.words, g.n_in, g.n_out = stream, torch.device("cpu"), True, 27, 1, n, n
    g.lists, g._reduced, g._reduced_streams, g._written, g._launches, g._tensors = None, {}, {}, set(), {}, {}
    g._allocate()
    return g, recorded, now


def test_reduced_masks_belong_to_the_streams_that_use_them(monkeypatch):
    """Built on one stream, first used on a second, used again on the first: the words of the kernels' tile
    heights lie in the block of the tables, others are recorded for every stream but their own."""
    from cumm_amd import torch_bridge as tb
    for n in (0, 1, 64, 65, 1000):
        g, recorded, now = _geometry(monkeypatch, tb, n)
        now[0] = 2
        g.used_on(2)
        at = {w: (g.reduced_address(w), 4 * max((n + w - 1) // w, 1)) for w in (64, 128, 32)}
        block = g._block.untyped_storage().data_ptr()
        assert recorded == [(block, 2)]
        spans = sorted([(a, a + size) for w, (a, size) in at.items() if w != 32] + [(g._ptr["order_fwd"], g._ptr["order_fwd"] + 4 * n)])
        assert block <= spans[0][0] and spans[-1][1] <= block + g._block.numel()
        assert all(x[1] <= y[0] for x, y in zip(spans, spans[1:]))
        assert not block <= at[32][0] < block + g._block.numel()
        now[0] = 1
        g.used_on(1)
        assert recorded[1:] == [(at[32][0], 1)]
        assert all(g.reduced_address(w) == a for w, (a, _) in at.items())


def test_a_reduced_mask_that_no_pass_has_written_is_zero(monkeypatch):
    import ctypes
    from cumm_amd import torch_bridge as tb
    g, _, _ = _geometry(monkeypatch, tb)
    g._block.fill_(0xA5)

    def words(w):
        t = g.reduced_mask_buffer(w)
        assert t.dtype == tv.uint32 and t.shape == [(1000 + w - 1) // w] and t.byte_pointer() == g.reduced_address(w)
        return (ctypes.c_uint32 * t.size).from_address(t.byte_pointer())
    for w in (64, 32):
        assert not any(words(w))
    g.reduced_address(128)      # (what a forward pass asks for, and fills)
    for w in (64, 32, 128):
        ctypes.memset(g.reduced_address(w), 7, 4)
        assert words(w)[0] == 0x07070707


def test_a_moved_call_refuses_tensors_on_another_device_than_the_tables(monkeypatch):
    """The tensors agree among themselves, the geometry lies elsewhere; and one tensor alone elsewhere."""
    from cumm_amd import torch_bridge as tb
    g, _, _ = _geometry(monkeypatch, tb)
    here, there = torch.empty(1), torch.empty(1, device="meta")
    assert tb._kind(g, ("fwd",), 1000, here, here)[0] == "fwd"
    for tensors in ((there, there, there), (here, there, here), (there, here, here)):
        with pytest.raises(ValueError, match="same device"):
            tb._kind(g, ("fwd",), 1000, *tensors)


def test_tables_that_were_handed_out_go_back_when_the_device_has_finished(monkeypatch):
    """A tv tensor of a table that outlives its geometry: the block is alive until the wait is over, and no
    wait is made for a geometry whose tables nobody took, nor while the stream is recorded."""
    from cumm_amd import torch_bridge as tb
    import gc
    import weakref
    waits, capturing = [], [False]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    for taken in (True, False):
        g, _, _ = _geometry(monkeypatch, tb)
        block = weakref.ref(g._block)
        monkeypatch.setattr(torch.cuda, "synchronize", lambda d: waits.append(block() is not None))
        table = g.indices_fwd_pos if taken else None
        if taken:
            assert table.byte_pointer() == g._ptr["indices_fwd_pos"] and g.indices_fwd_pos is table
        del g
        gc.collect()
        assert waits == [] and (block() is not None) == taken
        del table
        gc.collect()
        assert waits == ([True] if taken else []) and block() is None
        del waits[:]
    g, _, _ = _geometry(monkeypatch, tb)
    capturing[0] = g.order_fwd is not None
    del g
    gc.collect()
    assert waits == []


def test_a_table_by_position_is_completed_behind_the_construction(monkeypatch):
    """Read on another stream than the one that builds it, with another device current: the building stream is waited
    for, then the launch, on the geometry's device; not where either stream is being recorded.  A geometry that
    was built while its stream was recorded is completed at every read."""
    import contextlib
    from cumm_amd import torch_bridge as tb
    waited = []

    def fresh(n=1000):
        g, _, now = _geometry(monkeypatch, tb, n, stream=7)
        monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: type("S", (), {"synchronize": lambda self: waited.append(now[0])})())
        g._partial = frozenset(("indices_fwd_pos", "indices_bwd_pos"))
        now[0] = 9
        return g, now
    device, here, building = [None], [False], [False]

    @contextlib.contextmanager
    def on(d):
        device[0] = d
        yield
        device[0] = None
    monkeypatch.setattr(torch.cuda, "device", on)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: here[0])
    log, addresses = [], []

    class Library:
        def cumm_hip_stream_is_capturing(self, stream):
            assert stream == 7
            return building[0]

        def cumm_hip_stream_synchronize(self, stream):
            log.append(("wait", stream))
            return 0

        def cumm_hip_pairs_by_position(self, indices, order, kv, n, to, stream):
            assert device[0] == torch.device("cpu")
            addresses.append((indices, order, to))
            log.append(("write", stream))
            return 0
    monkeypatch.setattr(_capi, "_lib", Library())
    g, now = fresh()
    want = tuple(g._ptr[name] for name in ("indices_fwd", "order_fwd", "indices_fwd_pos"))
    for _ in range(2):      # (the second read finds it whole)
        assert g.indices_fwd_pos.byte_pointer() == g._ptr["indices_fwd_pos"]
        assert log == [("wait", 7), ("write", 9)] and waited == [9] and g._partial == {"indices_bwd_pos"}
        assert addresses == [want]
    del log[:], waited[:]
    g, now = fresh()
    now[0] = 7
    g.indices_fwd_pos
    assert log == [("write", 7)] and waited == [7]
    for here[0], building[0], left in ((True, False, 2), (False, True, 1)):
        del log[:], waited[:]
        g, now = fresh()
        g.indices_fwd_pos
        assert log == [("write", 9)] and waited == ([] if here[0] else [9]) and len(g._partial) == left
    building[0] = False
    del log[:], waited[:]
    g, now = fresh()
    g._recorded = True
    for trip in (1, 2):
        g.indices_fwd_pos
        assert log == [("wait", 7), ("write", 9)] * trip and len(g._partial) == 2


def test_pair_lists_wait_only_where_they_were_handed_out(monkeypatch):
    """The lists of a geometry with several mask words: the passes' own go back without a wait (their streams
    are recorded), those that somebody took keep the memory until the device has finished."""
    from cumm_amd import torch_bridge as tb
    import gc
    import weakref
    waits = []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    for taken in (True, False):
        g, recorded, now = _geometry(monkeypatch, tb)
        del g.lists
        g._list_block = torch.zeros((2, 27, 1000), dtype=torch.int32)
        g._lists = g._lists_over(g._list_block, torch.zeros(27, dtype=torch.int32).numpy())
        block = weakref.ref(g._list_block)
        monkeypatch.setattr(torch.cuda, "synchronize", lambda d: waits.append(block() is not None))
        now[0] = 2
        g.used_on(2)
        assert [s for _, s in recorded] == [2, 2] and recorded[1][0] == g._list_block.data_ptr()
        lists = g.lists if taken else None
        if taken:
            assert g.lists is lists and [t.byte_pointer() for t in lists[:2]] == [t.data_ptr() for t in g._list_block]
        del g
        gc.collect()
        assert waits == [] and (block() is not None) == taken
        del lists
        gc.collect()
        assert waits == ([True] if taken else []) and block() is None
        del waits[:]
    g, _, _ = _geometry(monkeypatch, tb)
    del g.lists
    assert g.lists is None


def test_a_remembered_call_refuses_tensors_on_another_device(monkeypatch):
    """A call that the geometry remembers takes addresses: the device of every tensor is looked at before each
    of them, in both passes - the first use on a geometry was checked, later ones were not."""
    from cumm_amd import torch_bridge as tb
    g, _, _ = _geometry(monkeypatch, tb)
    calls = []

    class Launch:
        tile_m = 64

        def __call__(self, stream, *a, **tensors):
            calls.append(tensors)

    class Known(dict):
        def get(self, key, default=None):
            return (Launch(), 256) if key[0] == "wgrad" else Launch()
    g._launches = Known()
    monkeypatch.setattr(tb._capi, "lib", lambda: None)
    x, w, b, y = torch.zeros(1000, 8).half(), torch.zeros(16, 27, 8).half(), torch.zeros(16).half(), torch.zeros(1000, 16).half()
    away = lambda t: t.to("meta")
    assert tb._SparseConvFunction.apply(x, w, b, g, False).shape == (1000, 16) and len(calls) == 1
    for tensors in ((away(x), w, b), (x, away(w), b), (x, w, away(b))):
        with pytest.raises(ValueError, match="same device"):
            tb._SparseConvFunction.apply(*tensors, g, False)
    assert len(calls) == 1
    ctx = type("Ctx", (), dict(geometry=g, relu=False, has_bias=False, tile_m=64, needs_input_grad=(True, True, False)))()

    def backward(x, w, y):
        ctx.saved_tensors = (x, w, None)
        return tb._SparseConvFunction.backward(ctx, y)
    backward(x, w, y)
    assert len(calls) == 3
    for tensors in ((away(x), w, y), (x, away(w), y), (x, w, away(y))):
        with pytest.raises(ValueError, match="same device"):
            backward(*tensors)
    assert len(calls) == 3


@pytest.mark.parametrize("error", [RuntimeError("g++ failed"), FileNotFoundError("g++")])
def test_a_machine_without_a_host_compiler_is_told_and_served(monkeypatch, tmp_path, error):
    from cumm_amd import build, torch_bridge as tb

    def fail(*a, **k):
        raise error
    monkeypatch.setattr(build, "TORCH_LIB", str(tmp_path / "_torch_native.so"))
    monkeypatch.setattr(build, "build_torch_native", fail)
    monkeypatch.setattr(tb, "_native_module", None)
    with pytest.warns(RuntimeWarning, match="g\\+\\+"):
        assert tb._native() is None
    assert tb._native() is None      # (and does not try again)


def test_a_native_half_of_other_sources_is_built_again(monkeypatch, tmp_path):
    """By what it was built from, not by its age: a file that came with an archive is as old as anything."""
    from cumm_amd import build
    source, lib = tmp_path / "torch_native.cpp", tmp_path / "_torch_native.so"
    source.write_text("one")
    monkeypatch.setattr(build, "TORCH_SRC", str(source))
    monkeypatch.setattr(build, "TORCH_LIB", str(lib))
    built = []

    def compiler(cmd, **k):
        built.append(cmd)
        with open(cmd[cmd.index("-o") + 1], "w") as f:
            f.write("..cumm_torch_native:" + [a for a in cmd if a.startswith("-DCUMM_STAMP=")][0].split('"')[1] + "..")
        return subprocess.CompletedProcess(cmd, 0, "")
    monkeypatch.setattr(build.subprocess, "run", compiler)
    for text, count in (("one", 1), ("one", 1), ("two", 2), ("two", 2)):
        source.write_text(text)
        os.utime(source, (0, 0))
        assert build.build_torch_native() == str(lib)
        assert len(built) == count, text
    monkeypatch.setattr(torch, "__version__", "another")
    build.build_torch_native()
    assert len(built) == 3


def test_builds_of_the_native_half_at_once_do_not_share_a_file(monkeypatch, tmp_path):
    """A build that ends while another one writes puts its own whole file in place; one that fails leaves nothing."""
    from cumm_amd import build
    monkeypatch.setattr(build, "TORCH_LIB", str(tmp_path / "_torch_native.so"))
    inside = []

    def compiler(cmd, **k):
        out = cmd[cmd.index("-o") + 1]
        with open(out, "w") as f:
            f.write("half")
        if not inside:
            inside.append(out)
            other = threading.Thread(target=build.build_torch_native, kwargs=dict(force=True))
            other.start()
            other.join()
            assert open(build.TORCH_LIB).read() == "whole"
        with open(out, "w") as f:
            f.write("whole")
        return subprocess.CompletedProcess(cmd, 0, "")
    monkeypatch.setattr(build.subprocess, "run", compiler)
    build.build_torch_native(force=True)
    assert open(build.TORCH_LIB).read() == "whole" and os.listdir(tmp_path) == ["_torch_native.so"]

    def failing(cmd, **k):
        compiler(cmd)
        return subprocess.CompletedProcess(cmd, 1, "no")
    monkeypatch.setattr(build.subprocess, "run", failing)
    with pytest.raises(RuntimeError, match="no"):
        build.build_torch_native(force=True)
    assert os.listdir(tmp_path) == ["_torch_native.so"]
