"""The pair-list weight gradient (wgrad_pairs.h) where its cuts fall: one step and less, one pair more
than a step, shares of the stream that end inside a list, empty lists, channel blocks with remainders,
row numbers out of range - against fp32 products of the same operands in numpy."""
import ctypes

import numpy as np
import pytest

from cumm_amd import _capi
from cumm_amd import tensorview as tv
from cumm_amd.gemm.main import GemmMainUnitTest, desp_to_c
from cumm_amd.tensorview.gemm import GemmParams, ShuffleStrideType
import helpers as H

torch = pytest.importorskip("torch")      # (before the library: one HIP runtime in the process)
pytestmark = pytest.mark.gpu

# the result is rounded once from fp32 sums: half a unit in the last place of the largest element, and
# the sums themselves to about 1e-5
TOL = {"f16": 2.0 ** -11 + 1e-4, "bf16": 2.0 ** -8 + 1e-4}


def _data(rng, shape, dtype):
    return H.to_storage(rng.normal(0, 1, size=shape).astype(np.float32), dtype)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("counts,k_out,c_in", [
    ([1], 8, 8), ([32], 64, 64), ([33, 0, 31], 72, 16), ([0, 0, 127, 128, 129], 64, 136), ([0], 16, 24),
    ([40000], 64, 64), ([9000, 0, 1, 20000, 5], 128, 72), ([300] * 125, 24, 40), ([2000] * 128, 64, 8)])
def test_pair_lists(counts, k_out, c_in, dtype):
    print("case wgrad_pairs", counts[:6], len(counts), k_out, c_in, dtype, flush=True)
    rng = np.random.default_rng(sum(counts) + k_out)
    lists, stride = len(counts), max(max(counts), 1) + 3
    rows_out, rows_in = 777, 1234
    dout, inp = _data(rng, (rows_out, k_out), dtype), _data(rng, (rows_in, c_in), dtype)
    po = rng.integers(0, rows_out, size=(lists, stride)).astype(np.int32)
    pi = rng.integers(0, rows_in, size=(lists, stride)).astype(np.int32)
    po[:, ::17], pi[:, 5::29] = -1, rows_in        # absent rows
    lib = _capi.lib()
    cnt = np.array(counts, np.int32)
    need = int(lib.cumm_hip_wgrad_pairs_workspace(cnt.ctypes.data, lists, k_out, c_in))
    ws = H.dev(np.full(max(need // 4, 4), np.nan, np.float32), "f32")
    dw = H.dev(_data(rng, (k_out, lists, c_in), dtype), dtype)
    d_out, d_in, d_po, d_pi = H.dev(dout, dtype), H.dev(inp, dtype), H.dev(po, "i32"), H.dev(pi, "i32")
    got = []
    for _ in range(2):
        _capi.check(lib.cumm_hip_wgrad_pairs(dw.byte_pointer(), d_out.byte_pointer(), d_in.byte_pointer(), d_po.byte_pointer(),
                                             d_pi.byte_pointer(), cnt.ctypes.data, lists, stride, rows_out, rows_in, k_out, c_in,
                                             H.TV_DTYPE[dtype], ws.byte_pointer(), ws.nbytes, 0))
        got.append(H.as_f32(H.host(dw), dtype))
    f_out, f_in = H.as_f32(dout, dtype), H.as_f32(inp, dtype)
    ref = np.zeros((k_out, lists, c_in), np.float32)
    for r, n in enumerate(counts):
        ok = (po[r, :n] >= 0) & (pi[r, :n] < rows_in)
        ref[:, r] = f_out[po[r, :n][ok]].T @ f_in[pi[r, :n][ok]]
    assert np.array_equal(got[0], got[1])          # a fixed order of the sums
    scale = max(np.abs(ref).max(), 1.0)
    assert np.abs(got[0] - ref).max() <= TOL[dtype] * scale
    for r, n in enumerate(counts):
        if n == 0:
            assert not got[0][:, r].any()


@pytest.mark.parametrize("pairs", [255, 256, 1000, 33000])
@pytest.mark.parametrize("dtype,out", [("f16", "f16"), ("bf16", "f32")])
def test_shuffle_ab_epilogue_on_either_side_of_the_dispatch(pairs, dtype, out):
    """alpha, beta with a separate D, rows wider than the operand, ReLU, f32 results: the tiled kernel
    below 256 pairs, the pair-list kernel from there on."""
    from cumm_amd.tensorview.gemm import Activation
    print("case shuffle_ab", pairs, dtype, out, flush=True)
    rng = np.random.default_rng(pairs)
    rows, m, n = 5000, 72, 136
    a, b = _data(rng, (rows, m), dtype), _data(rng, (rows, n), dtype)
    ai, bi = (rng.integers(0, rows, size=pairs).astype(np.int32) for _ in range(2))
    d = _data(rng, (m, n), out) if out != "f32" else rng.normal(0, 1, size=(m, n)).astype(np.float32)
    p = GemmParams()
    p.algo_desp = H.find_gemm_desp(dtype, ShuffleStrideType.ShuffleAB, 64, 64, True, False, dtype_c=out)
    p.a, p.b = H.dev(a, dtype), H.dev(b, dtype)
    p.c = tv.zeros([m, n], H.TV_DTYPE[out], 0)
    p.d = H.dev(d, out)
    p.a_inds, p.b_inds = H.dev(ai, "i32"), H.dev(bi, "i32")
    p.alpha, p.beta, p.act_type = 0.25, 2.0, Activation.ReLU
    GemmMainUnitTest.matmul2(p)
    ref = np.maximum(0.25 * (H.as_f32(a, dtype)[ai].T @ H.as_f32(b, dtype)[bi]) + 2.0 * (H.as_f32(d, out) if out != "f32" else d), 0)
    got = H.host(p.c) if out == "f32" else H.as_f32(H.host(p.c), out)
    tol = 1e-5 * np.sqrt(pairs) if out == "f32" else TOL[out]
    assert np.abs(got - ref).max() <= tol * max(np.abs(ref).max(), 1.0)
    cd = desp_to_c(p.algo_desp)
    assert (int(_capi.lib().cumm_hip_query_gemm_optional_workspace(ctypes.byref(cd), m, n, pairs)) > 0) == (pairs >= 256)


@pytest.mark.parametrize("kv,wide", [(27, True), (130, False), (130, True)])
def test_backward_weight_of_strided_rows_and_of_more_offsets_than_one_call_takes(kv, wide):
    """Features and gradients that are columns of wider tensors, and more than 128 offsets: one product per
    offset, with the results of whole tensors."""
    from types import SimpleNamespace
    from cumm_amd.conv import native
    print("case backward_weight", kv, wide, flush=True)
    rng = np.random.default_rng(kv)
    rows, k_out, c_in, most = 600, 24, 40, 300
    dout, inp = _data(rng, (rows, k_out + 8 * wide), "f16"), _data(rng, (rows, c_in + 16 * wide), "f16")
    counts = rng.integers(0, most, size=kv).astype(np.int32)
    counts[3] = 0
    po, pi = (rng.integers(0, rows, size=(kv, most)).astype(np.int32) for _ in range(2))
    view = lambda a, n: H.dev(a, "f16").slice_axis(1, 0, n) if wide else H.dev(a, "f16")
    dw = H.dev(_data(rng, (k_out, kv, c_in), "f16"), "f16")
    lists = SimpleNamespace(pair_in=H.dev(pi, "i32"), pair_out=H.dev(po, "i32"), counts=counts)
    native.backward_weight(view(dout, k_out), view(inp, c_in), dw, lists)
    got = H.as_f32(H.host(dw), "f16")
    f_out, f_in = H.as_f32(dout, "f16")[:, :k_out], H.as_f32(inp, "f16")[:, :c_in]
    ref = np.stack([f_out[po[r, :n]].T @ f_in[pi[r, :n]] for r, n in enumerate(counts)], axis=1)
    assert np.abs(got - ref).max() <= TOL["f16"] * max(np.abs(ref).max(), 1.0)


@pytest.mark.parametrize("first", ["recorded", "eager"])
def test_shuffle_ab_recorded_into_a_graph(first):
    """Nothing is allocated while a stream is recorded, and a graph keeps its results when the parameter
    object it was recorded from is gone."""
    print("case shuffle_ab graph", first, flush=True)
    rng = np.random.default_rng(3)
    rows, m, n, pairs = 2000, 64, 72, 1000
    a, b = _data(rng, (rows, m), "f16"), _data(rng, (rows, n), "f16")
    ai, bi = (rng.integers(0, rows, size=pairs).astype(np.int32) for _ in range(2))
    c = tv.zeros([m, n], tv.float16, 0)
    p = GemmParams()
    p.algo_desp = H.find_gemm_desp("f16", ShuffleStrideType.ShuffleAB, 64, 64, True, False)
    p.a, p.b, p.c, p.a_inds, p.b_inds = H.dev(a, "f16"), H.dev(b, "f16"), c, H.dev(ai, "i32"), H.dev(bi, "i32")
    keep = (p.a, p.b, p.a_inds, p.b_inds)
    if first == "eager":
        GemmMainUnitTest.matmul2(p)
    warm = GemmParams()      # (loads the kernel that the graph will hold)
    warm.algo_desp = p.algo_desp
    warm.a, warm.b, warm.c = p.a, p.b, c
    warm.a_inds, warm.b_inds = p.a_inds.slice_first_axis(0, 100), p.b_inds.slice_first_axis(0, 100)
    GemmMainUnitTest.matmul2(warm)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        p.stream = torch.cuda.current_stream().cuda_stream
        GemmMainUnitTest.matmul2(p)
    # (a workspace that the graph used would be in p's prepared arguments: it has none)
    ref = H.as_f32(a, "f16")[ai].T @ H.as_f32(b, "f16")[bi]
    del p
    for _ in range(3):
        c.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.abs(H.as_f32(H.host(c), "f16") - ref).max() <= TOL["f16"] * np.abs(ref).max()
    del keep


@pytest.mark.parametrize("first", ["recorded", "eager"])
def test_all_offsets_recorded_into_a_graph(first):
    """A graph that outlives the plan it was recorded from, whose own workspace others use afterwards."""
    from types import SimpleNamespace
    from cumm_amd.conv import native
    print("case all offsets graph", first, flush=True)
    rng = np.random.default_rng(8)
    rows, k_out, c_in, most, counts = 600, 64, 72, 300, np.array([300, 0, 257], np.int32)
    dout, inp = _data(rng, (rows, k_out), "f16"), _data(rng, (rows, c_in), "f16")
    po, pi = (rng.integers(0, rows, size=(3, most)).astype(np.int32) for _ in range(2))
    lists = SimpleNamespace(pair_in=H.dev(pi, "i32"), pair_out=H.dev(po, "i32"), counts=counts)
    operands = (H.dev(dout, "f16"), H.dev(inp, "f16"), tv.zeros([k_out, 3, c_in], tv.float16, 0))
    ref = np.stack([H.as_f32(dout, "f16")[po[r, :n]].T @ H.as_f32(inp, "f16")[pi[r, :n]] for r, n in enumerate(counts)], axis=1)
    few, _ = _shuffle_ab(np.random.default_rng(6), 2000, 64, 72, 100)      # (loads the kernel that the graph will hold)
    GemmMainUnitTest.matmul2(few)
    side = torch.cuda.Stream()
    plan = native.plan_backward_weight(*operands, lists, stream=side.cuda_stream)
    if first == "eager":
        plan()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        plan()
    del plan
    for _ in range(3):
        other, want = _shuffle_ab(rng, 2000, 64, 72, 1000)
        operands[2].zero_()
        torch.cuda.synchronize()
        other.stream = side.cuda_stream
        graph.replay()
        GemmMainUnitTest.matmul2(other)
        torch.cuda.synchronize()
        for got, r in ((operands[2], ref), (other.c, want)):
            assert np.abs(H.as_f32(H.host(got), "f16") - r).max() <= TOL["f16"] * np.abs(r).max()


def _shuffle_ab(rng, rows, m, n, pairs):
    a, b = _data(rng, (rows, m), "f16"), _data(rng, (rows, n), "f16")
    ai, bi = (rng.integers(0, rows, size=pairs).astype(np.int32) for _ in range(2))
    p = GemmParams()
    p.algo_desp = H.find_gemm_desp("f16", ShuffleStrideType.ShuffleAB, 64, 64, True, False)
    p.a, p.b, p.a_inds, p.b_inds = H.dev(a, "f16"), H.dev(b, "f16"), H.dev(ai, "i32"), H.dev(bi, "i32")
    p.c = tv.zeros([m, n], tv.float16, 0)
    return p, H.as_f32(a, "f16")[ai].T @ H.as_f32(b, "f16")[bi]


@pytest.mark.parametrize("entry,used", [("cumm_hip_gemm", False), ("cumm_hip_gemm_in_workspace", True)])
def test_one_slice_uses_a_workspace_only_where_the_caller_says_so(entry, used):
    """A workspace passed along with split_k_slices == 1, as a caller of several streams may share it."""
    print("case shuffle_ab workspace", entry, flush=True)
    m, n, pairs = 64, 136, 5000
    p, ref = _shuffle_ab(np.random.default_rng(4), 3000, m, n, pairs)
    lib, cd = _capi.lib(), desp_to_c(p.algo_desp)
    ws = H.dev(np.full(int(lib.cumm_hip_query_gemm_optional_workspace(ctypes.byref(cd), m, n, pairs)), 0xA5, np.uint8), "u8")
    args = _capi.GemmArgs()
    args.m, args.n, args.k, args.alpha, args.split_k_slices = m, n, pairs, 1.0, 1
    args.ptr_A, args.ptr_B, args.ptr_C = p.a.byte_pointer(), p.b.byte_pointer(), p.c.byte_pointer()
    args.stride_A, args.stride_B, args.stride_C = m, n, n
    args.indiceA, args.indiceBorC = p.a_inds.byte_pointer(), p.b_inds.byte_pointer()
    args.workspace, args.workspace_bytes = ws.byte_pointer(), ws.nbytes
    args.rows_A, args.rows_B, args.rows_C = 3000, 3000, m
    _capi.check(getattr(lib, entry)(ctypes.byref(cd), ctypes.byref(args), 0))
    assert np.abs(H.as_f32(H.host(p.c), "f16") - ref).max() <= TOL["f16"] * np.abs(ref).max()
    assert bool((H.host(ws) != 0xA5).any()) == used


def test_a_validated_call_recorded_into_a_graph_leaves_its_workspace_alone():
    """The call is validated on the stream that is recorded afterwards, the parameter object stays as it is."""
    print("case shuffle_ab graph validated", flush=True)
    p, ref = _shuffle_ab(np.random.default_rng(5), 2000, 64, 72, 1000)
    few, _ = _shuffle_ab(np.random.default_rng(6), 2000, 64, 72, 100)      # (loads the kernel that the graph will hold)
    GemmMainUnitTest.matmul2(few)
    side = torch.cuda.Stream()
    p.stream = side.cuda_stream
    GemmMainUnitTest.matmul2(p)
    kept = p.__dict__["_prepared"]
    workspace = kept[6]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        GemmMainUnitTest.matmul2(p)
    assert p.__dict__["_prepared"] is kept and workspace.nbytes > 0
    for _ in range(3):
        workspace.fill_int_(0x5A)
        p.c.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.abs(H.as_f32(H.host(p.c), "f16") - ref).max() <= TOL["f16"] * np.abs(ref).max()
        assert bool((H.host(workspace) == 0x5A).all())
        GemmMainUnitTest.matmul2(p)      # the eager call still uses it
        torch.cuda.synchronize()
        assert bool((H.host(workspace) != 0x5A).any())


def test_new_parameter_objects_allocate_no_workspace_of_their_own(monkeypatch):
    """A loop over offsets with an object per call, and one object that is given new index lists."""
    print("case shuffle_ab new objects", flush=True)
    p, ref = _shuffle_ab(np.random.default_rng(7), 3000, 64, 72, 4000)
    real, calls = _capi.lib(), []

    class Counting:
        def __getattr__(self, name):
            if name in ("cumm_hip_malloc", "cumm_hip_free"):
                calls.append(name)
            return getattr(real, name)

    def again():
        q = GemmParams()
        q.algo_desp = p.algo_desp
        q.a, q.b, q.c, q.a_inds, q.b_inds = p.a, p.b, p.c, p.a_inds, p.b_inds
        GemmMainUnitTest.matmul2(q)
    full = p.a_inds, p.b_inds
    GemmMainUnitTest.matmul2(p)
    again()
    monkeypatch.setattr(_capi, "_lib", Counting())
    for pairs in (4000, 300, 4000):
        again()
        p.a_inds, p.b_inds = (t.slice_first_axis(0, pairs) for t in full)
        GemmMainUnitTest.matmul2(p)
    monkeypatch.setattr(_capi, "_lib", real)
    assert calls == []
    assert np.abs(H.as_f32(H.host(p.c), "f16") - ref).max() <= TOL["f16"] * np.abs(ref).max()


def test_a_plan_of_single_products_on_other_tensors_and_another_stream():
    """Columns of wider tensors: the plan's second run, on tensors of its own and a second stream."""
    from types import SimpleNamespace
    from cumm_amd.conv import native
    print("case weight steps rebind", flush=True)
    rng = np.random.default_rng(8)
    kv, rows, k_out, c_in, most = 5, 900, 24, 40, 3000
    counts = np.array([3000, 0, 17, 257, 1500], np.int32)
    po, pi = (rng.integers(0, rows, size=(kv, most)).astype(np.int32) for _ in range(2))
    lists = SimpleNamespace(pair_in=H.dev(pi, "i32"), pair_out=H.dev(po, "i32"), counts=counts)
    sets = []
    for _ in range(2):
        dout, inp = _data(rng, (rows, k_out + 8), "f16"), _data(rng, (rows, c_in + 16), "f16")
        f_out, f_in = H.as_f32(dout, "f16")[:, :k_out], H.as_f32(inp, "f16")[:, :c_in]
        ref = np.stack([f_out[po[r, :n]].T @ f_in[pi[r, :n]] for r, n in enumerate(counts)], axis=1)
        sets.append((H.dev(dout, "f16").slice_axis(1, 0, k_out), H.dev(inp, "f16").slice_axis(1, 0, c_in),
                     H.dev(_data(rng, (k_out, kv, c_in), "f16"), "f16"), ref))
    plan = native.plan_backward_weight(*sets[0][:3], lists)
    assert isinstance(plan, native.WeightSteps)
    side = torch.cuda.Stream()
    plan()
    plan()
    torch.cuda.synchronize()
    plan.rebind(*(t.byte_pointer() for t in sets[1][:3]), side.cuda_stream)
    torch.cuda.synchronize()
    for _, _, dw, ref in sets:
        assert np.abs(H.as_f32(H.host(dw), "f16") - ref).max() <= TOL["f16"] * np.abs(ref).max()


@pytest.mark.parametrize("k_out,c_in,pairs", [(576, 256, 400), (576, 520, 3000), (1024, 1024, 384), (1000, 1016, 5000), (2048, 136, 700)])
def test_more_channel_blocks_than_a_share_fits_one_xcd(k_out, c_in, pairs):
    """36 to 256 blocks of 64 x 64 channels: fewer than eight shares of the pairs, one for the largest."""
    print("case wgrad_pairs blocks", k_out, c_in, pairs, flush=True)
    p, ref = _shuffle_ab(np.random.default_rng(pairs), 2500, k_out, c_in, pairs)
    GemmMainUnitTest.matmul2(p)
    cd = desp_to_c(p.algo_desp)
    assert int(_capi.lib().cumm_hip_query_gemm_optional_workspace(ctypes.byref(cd), k_out, c_in, pairs)) > 0
    assert int(_capi.lib().cumm_hip_query_gemm_optional_workspace(ctypes.byref(cd), k_out, c_in, 383)) == 0
    assert np.abs(H.as_f32(H.host(p.c), "f16") - ref).max() <= TOL["f16"] * np.abs(ref).max()
