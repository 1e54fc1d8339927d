"""cumm_hip_sparse_conv_more: what a training program wants of the convolution launches beyond the reference's
argument block."""
import ctypes

import numpy as np
import pytest

import helpers as H
from cumm_amd import _capi, pairs, synth
from cumm_amd import tensorview as tv
from cumm_amd.conv.main import ConvMainUnitTest
from cumm_amd.tensorview.gemm import Activation, ConvOpType, ConvParams

pytestmark = pytest.mark.gpu


def _again(p, **more):
    """The call that ``p`` has just made, once more with ``more``."""
    prep = p.__dict__["_prepared"]
    extra = _capi.SparseConvMore(**more)
    _capi.check(_capi.lib().cumm_hip_sparse_conv_more(ctypes.byref(prep[4]), ctypes.byref(prep[5]), ctypes.byref(extra), p.stream))
    _capi.check(_capi.lib().cumm_hip_device_synchronize())


@pytest.mark.parametrize("channels,tile", [(64, (64, 64)), (32, (64, 64)), (64, (128, 64)), (128, (128, 128)), (72, (64, 128))])
@pytest.mark.parametrize("hint", [0, -1])
def test_write_empty(channels, tile, hint):
    """Backward-input of a stride-2 layer whose inputs on the last plane of an axis feed no output: their rows come
    back as zeros instead of being left alone, the others with the same bits (128-row runs of a mixed launch that are
    half empty among them)."""
    print("case write empty", channels, tile, hint, flush=True)
    rng, dtype, k_out = np.random.default_rng(12), "f16", 64
    grid = (12, 40, 36)
    coords = synth.clustered_voxels(rng, 2500, grid, 6, sigma=3.0)
    zz, yy = np.meshgrid(np.arange(grid[0]), np.arange(grid[1]), indexing="ij")
    plane = np.stack([np.zeros(zz.size, np.int64), zz.ravel(), yy.ravel(), np.full(zz.size, grid[2] - 1)], axis=1)
    coords = np.unique(np.concatenate([coords, plane.astype(np.int32)]), axis=0).astype(np.int32)
    pt = pairs.sparse_conv_pairs(coords, grid, padding=(0, 0, 0))
    n_in, n_out = coords.shape[0], pt.indices_fwd.shape[1]
    ms, order = pairs.sort_by_mask(pt.mask_bwd)
    empty = order[:int((ms == 0).sum()) // 128 * 128]
    assert len(empty) >= 256
    w = H.to_storage(rng.normal(0, 0.05, size=(k_out, 27, channels)).astype(np.float32), dtype)
    dout = H.to_storage(rng.normal(0, 1, size=(n_out, k_out)).astype(np.float32), dtype)
    p = ConvParams(3, ConvOpType.BackwardInput)
    p.conv_algo_desp = H.find_conv_desp(dtype, ConvOpType.BackwardInput, *tile)
    p.input = H.dev(H.to_storage(np.full((n_in, channels), 7.0, np.float32), dtype), dtype)
    p.weight, p.output = H.dev(w, dtype), H.dev(dout, dtype)
    p.indices, p.mask, p.mask_argsort = H.dev(pt.indices_bwd, "i32"), H.dev(ms, "u32"), H.dev(order, "i32")
    p.light_prefix = hint
    ConvMainUnitTest.implicit_gemm2(p)
    base = H.as_f32(H.host(p.input), dtype)
    assert (base[empty] == 7.0).all()
    _again(p, write_empty=1)
    got = H.as_f32(H.host(p.input), dtype)
    assert (got[np.asarray(pt.mask_bwd) == 0] == 0.0).all()
    live = np.asarray(pt.mask_bwd) != 0
    np.testing.assert_array_equal(got[live], base[live])


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("tile", [(64, 64), (128, 128)])
@pytest.mark.parametrize("act", [Activation.None_, Activation.ReLU])
@pytest.mark.parametrize("with_bias", [False, True])
def test_special_values_through_the_epilogue(dtype, tile, act, with_bias):
    """Results that are NaN, infinite, overflow in the rounding or are a negative zero: the identity as weight of the
    one kernel offset, so that a result is a feature times alpha plus the bias, rounded once."""
    print("case special values", dtype, tile, act, with_bias, flush=True)
    rng, n, c = np.random.default_rng(3), 300, 128 if tile[1] == 128 else 64
    x = rng.normal(0, 1, size=(n, c)).astype(np.float32)
    for i, v in enumerate((np.nan, np.inf, -np.inf, 0.0, -0.0, 65000.0, -65000.0, 3.3e38, -3.3e38)):
        x[i * 7 % n, i::9] = v if dtype == "bf16" or abs(v) < 65504 or not np.isfinite(v) else 1.0
    feat, bias = H.to_storage(x, dtype), H.to_storage(rng.normal(0, 1, size=c).astype(np.float32), dtype)
    p = ConvParams(3, ConvOpType.Forward)
    p.conv_algo_desp = H.find_conv_desp(dtype, ConvOpType.Forward, *tile)
    w = np.zeros((c, 1, c), np.float32)
    p.input, p.output = H.dev(feat, dtype), tv.zeros([n, c], H.TV_DTYPE[dtype], 0)
    w[np.arange(c), 0, np.arange(c)] = 1.0
    clean = np.nan_to_num(H.as_f32(feat, dtype), nan=0.0, posinf=0.0, neginf=0.0)
    p.weight = H.dev(H.to_storage(w, dtype), dtype)
    rows = np.arange(n, dtype=np.int32)
    p.indices, p.mask, p.mask_argsort = H.dev(rows[None], "i32"), H.dev(np.ones(n, np.uint32), "u32"), H.dev(rows, "i32")
    p.alpha, p.act_type = -1.5, act
    if with_bias:
        p.bias, p.beta = H.dev(bias, dtype), 1.0
    ConvMainUnitTest.implicit_gemm2(p)
    # (0 * inf and 0 * NaN of the other columns make all of such a row NaN before the epilogue)
    whole = np.isfinite(H.as_f32(feat, dtype)).all(axis=1, keepdims=True)
    acc = np.where(whole, clean, np.float32(np.nan))
    with np.errstate(over="ignore", invalid="ignore"):
        want = (acc.astype(np.float64) * -1.5 + (H.as_f32(bias, dtype) if with_bias else 0)).astype(np.float32)      # (the fused form)
        if act == Activation.ReLU:
            want = np.where(want > 0, want, np.float32(0))
        want = H.to_storage(want, dtype)
    got = H.host(p.output)
    a, b = got.view(np.uint16), want.view(np.uint16)
    nan = np.isnan(H.as_f32(want, dtype))
    np.testing.assert_array_equal(np.isnan(H.as_f32(got, dtype)), nan)
    assert nan.any() == (act == Activation.None_)
    if dtype == "bf16":
        assert (a[nan] == 0x7FFF).all()
    np.testing.assert_array_equal(a[~nan] & 0x7FFF, b[~nan] & 0x7FFF)
    keep = ~nan & ((a & 0x7FFF) != 0) if act == Activation.None_ else ~nan      # (the sign of a zero sum is the matrix unit's)
    np.testing.assert_array_equal(a[keep], b[keep])


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("n,cin,k_out,slices,ordered", [
    (1, 8, 8, 32, False),            # one row
    (3000, 64, 64, 32, False),       # lists, a copy of the image per eighth of the units
    (3000, 64, 64, 32, True),        # lists, slots in a fixed order
    (2500, 136, 72, 32, False),      # units of 128 x 128 channels; a group of bias sums that is half empty
    (2500, 136, 72, 32, True),
    (3000, 64, 64, 1, False),        # the tiled kernel
    (66000, 8, 1000, 32, False),     # sums in two stages
])
@pytest.mark.parametrize("relu", [False, True])
def test_gate_and_sums_of_a_weight_gradient(dtype, n, cin, k_out, slices, ordered, relu):
    """Gate and bias gradient in the launches of the weight gradient, with the table by row and by position, against
    numpy.  Small whole numbers: every sum is
    exact in fp32 whatever its order, and is rounded once."""
    print("case gate and sums", dtype, n, cin, k_out, slices, ordered, relu, flush=True)
    rng = np.random.default_rng(n + cin)
    grad, out, x = (rng.integers(-1, 2, size=(n, c)).astype(np.float32) for c in (k_out, k_out, cin))
    kv = 2
    indices = np.stack([rng.permutation(n), np.where(rng.random(n) < 0.5, rng.permutation(n), -1)]).astype(np.int32)
    mask = (1 + 2 * (indices[1] >= 0)).astype(np.uint32)
    ms, order = pairs.sort_by_mask(mask)
    width = 64
    red = np.bitwise_or.reduceat(ms, np.arange(0, n, width)).astype(np.uint32)
    gated = np.where(out > 0, grad, np.float32(0)) if relu else grad
    dw = np.stack([gated.T @ x[indices[0]], gated[indices[1] >= 0].T @ x[indices[1][indices[1] >= 0]]], axis=1)

    p = ConvParams(3, ConvOpType.BackwardWeight)
    p.conv_algo_desp = H.find_conv_desp(dtype, ConvOpType.BackwardWeight, 64, 64, split_k_parallel=True)
    d_grad, d_out = H.dev(H.to_storage(grad, dtype), dtype), H.dev(H.to_storage(out, dtype), dtype)
    d_gated = H.dev(H.to_storage(np.full_like(grad, 9.0), dtype), dtype) if relu else d_grad
    p.input, p.output = H.dev(H.to_storage(x, dtype), dtype), d_gated
    p.weight = tv.zeros([k_out, kv, cin], H.TV_DTYPE[dtype], 0)
    p.indices, p.mask, p.mask_argsort = H.dev(indices, "i32"), H.dev(red, "u32"), H.dev(order, "i32")
    p.mask_width, p.split_k_slices, p.deterministic = width, slices, ordered
    ConvMainUnitTest.implicit_gemm2(p)      # (of whatever d_gated holds)
    sums = tv.zeros([k_out], H.TV_DTYPE[dtype], 0)
    need = int(_capi.lib().cumm_hip_column_sum_workspace(n, k_out))
    ws = tv.zeros([need], tv.uint8, 0)
    gs = _capi.GateSums(gated=d_gated.byte_pointer() if relu else None, sums=sums.byte_pointer(), grad=d_grad.byte_pointer(),
                        out=d_out.byte_pointer() if relu else None, rows=n, channels=k_out, workspace=ws.byte_pointer(),
                        workspace_bytes=need)
    by_position = H.dev(np.ascontiguousarray(indices[:, order]), "i32")
    for more in ({}, {"by_position": by_position.byte_pointer()}):
        _again(p, sums=ctypes.addressof(gs), **more)
        np.testing.assert_array_equal(H.as_f32(H.host(d_gated), dtype), gated)
        np.testing.assert_array_equal(H.host(sums).view(np.uint16), H.to_storage(gated.sum(axis=0), dtype).view(np.uint16))
        np.testing.assert_array_equal(H.as_f32(H.host(p.weight), dtype), H.as_f32(H.to_storage(dw, dtype), dtype))
        for t in (sums, p.weight) + ((d_gated,) if relu else ()):
            _capi.check(_capi.lib().cumm_hip_memset(t.byte_pointer(), 0x55, t.size * t.itemsize, None))


def test_gate_and_sums_are_of_the_gradient_of_the_call():
    """Sums of another tensor than the one that the call reads are refused, as is a pass without a weight gradient."""
    lib, ws = _capi.lib(), tv.zeros([1 << 16], tv.uint8, 0)
    t = [tv.zeros([64, 64], tv.float16, 0) for _ in range(3)]
    gs = _capi.GateSums(gated=None, sums=ws.byte_pointer(), grad=t[2].byte_pointer(), rows=64, channels=64,
                        workspace=ws.byte_pointer() + 4096, workspace_bytes=1 << 15)
    for op, parallel in ((ConvOpType.BackwardWeight, True), (ConvOpType.Forward, False)):
        p = ConvParams(3, op)
        p.conv_algo_desp = H.find_conv_desp("f16", op, 64, 64, split_k_parallel=parallel)
        p.input, p.output, p.weight = t[0], t[1], tv.zeros([64, 1, 64], tv.float16, 0)
        p.indices, p.mask, p.mask_argsort = (H.dev(np.arange(64, dtype=np.int32)[None], "i32"), H.dev(np.ones(64, np.uint32), "u32"),
                                             H.dev(np.arange(64, dtype=np.int32), "i32"))
        if parallel:
            p.mask, p.mask_width, p.split_k_slices = H.dev(np.ones(1, np.uint32), "u32"), 64, 4
        ConvMainUnitTest.implicit_gemm2(p)
        with pytest.raises(ValueError):
            _again(p, sums=ctypes.addressof(gs))


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("ksize,cin,k_out,tile,n,hint", [
    (3, 64, 64, (64, 64), 40000, 0), (3, 64, 64, (64, 64), 40000, -1),     # tile shapes mixed, and one
    (3, 16, 24, (64, 64), 700, 0), (3, 64, 8, (64, 64), 700, 0),            # two groups of waves; one byte a position
    (3, 64, 72, (128, 64), 700, 0), (3, 64, 136, (64, 128), 700, 0),        # a last group of one byte
    (3, 64, 256, (128, 128), 700, 0), (3, 136, 128, (128, 128), 700, 0),
    (5, 32, 40, (64, 64), 700, 0), (5, 32, 128, (128, 128), 700, 0),        # several mask words
    (3, 520, 64, (64, 64), 700, 0),                                         # kernels that leave the gate to another one
])
def test_gate_of_a_forward_pass(dtype, ksize, cin, k_out, tile, n, hint):
    """The bits that a ReLU layer leaves are those of its output; a gradient gated by them is what the output gives, its
    sums too: of whole numbers, exact in any order, and in one order of the rows of any numbers."""
    print("case gate", dtype, ksize, cin, k_out, tile, n, hint, flush=True)
    rng, lib = np.random.default_rng(k_out), _capi.lib()
    coords, grid = H.small_cloud(5, n, grid=(20, 90, 90), clusters=12, sigma=6.0)
    n, kv = coords.shape[0], ksize ** 3
    table = pairs.subm_pairs_device(H.dev(coords, "i32"), grid, (ksize,) * 3)
    p = ConvParams(3, ConvOpType.Forward)
    if kv > 32:
        p.conv_algo_desp = H.find_conv_desp(dtype, ConvOpType.Forward, *tile, dynamic_mask=True)
        p.mask, p.mask_argsort = pairs.sort_by_mask_words_device(pairs.masks_from_pairs_device(table.indices_fwd))
        p.mask_int_count = (kv + 31) // 32
    else:
        p.conv_algo_desp = H.find_conv_desp(dtype, ConvOpType.Forward, *tile)
        p.mask, p.mask_argsort = pairs.sort_by_mask_device(table.mask_fwd, (1 << kv) - 1, by_offset_count=True)
    p.input = H.dev(H.to_storage(rng.normal(0, 1, size=(n, cin)).astype(np.float32), dtype), dtype)
    p.weight = H.dev(H.to_storage(rng.normal(0, 0.05, size=(k_out, kv, cin)).astype(np.float32), dtype), dtype)
    p.output, p.bias, p.beta = tv.zeros([n, k_out], H.TV_DTYPE[dtype], 0), H.dev(H.to_storage(rng.normal(0, 0.3, size=k_out).astype(np.float32), dtype), dtype), 1.0
    p.act_type, p.indices, p.light_prefix = Activation.ReLU, table.indices_fwd, hint
    ConvMainUnitTest.implicit_gemm2(p)
    before, groups = H.host(p.output).copy(), (k_out + 63) // 64
    d_gate = tv.from_numpy(np.full((groups, n, 8), 0xA5, np.uint8)).cuda()
    _again(p, gate=d_gate.byte_pointer())
    out, order = H.host(p.output), H.host(p.mask_argsort)
    np.testing.assert_array_equal(out.view(np.uint16), before.view(np.uint16))
    want = np.packbits(H.as_f32(out, dtype)[order] > 0, axis=1, bitorder="little")      # [n, k_out / 8]
    got = H.host(d_gate).transpose(1, 0, 2).reshape(n, groups * 8)[:, :k_out // 8]
    np.testing.assert_array_equal(got, want)

    need = int(lib.cumm_hip_column_sum_workspace(n, k_out))
    in_order = p.mask_argsort.byte_pointer()
    sources = ({"out": p.output.byte_pointer()}, {"out": p.output.byte_pointer(), "order": in_order},
               {"gate": d_gate.byte_pointer(), "order": in_order})
    for grad in (rng.normal(0, 1, size=(n, k_out)).astype(np.float32), rng.integers(-2, 3, size=(n, k_out)).astype(np.float32)):
        whole = bool((grad == np.rint(grad)).all())
        d_grad, ws = H.dev(H.to_storage(grad, dtype), dtype), tv.zeros([need], tv.uint8, 0)
        got = []
        for source in sources:
            gated, sums = tv.zeros([n, k_out], H.TV_DTYPE[dtype], 0), tv.zeros([k_out], H.TV_DTYPE[dtype], 0)
            gs = _capi.GateSums(gated=gated.byte_pointer(), sums=sums.byte_pointer(), grad=d_grad.byte_pointer(), rows=n, channels=k_out,
                                workspace=ws.byte_pointer(), workspace_bytes=need, **source)
            _capi.check(lib.cumm_hip_gate_sums(ctypes.byref(gs), int(H.TV_DTYPE[dtype]), None))
            _capi.check(lib.cumm_hip_device_synchronize())
            got.append((H.host(gated).view(np.uint16), H.host(sums).view(np.uint16)))
        for one, two in ((0, 1), (1, 2)):
            np.testing.assert_array_equal(got[one][0], got[two][0])
            if whole or one == 1:
                np.testing.assert_array_equal(got[one][1], got[two][1])
        np.testing.assert_array_equal(got[0][0] & 0x7FFF != 0, (H.as_f32(out, dtype) > 0) & (H.to_storage(grad, dtype).view(np.uint16) & 0x7FFF != 0))


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("rows,channels", [(1, 64), (700, 64), (700, 136), (40000, 72)])
def test_positions_that_name_no_row(dtype, rows, channels):
    """A few positions of the order lie outside the rows: they are passed over, and the rows that nobody names are left
    alone."""
    print("case no row", dtype, rows, channels, flush=True)
    rng, lib = np.random.default_rng(rows), _capi.lib()
    order = rng.permutation(rows).astype(np.int32)
    outside = np.unique(rng.integers(0, rows, size=min(rows, 9)))
    named = np.ones(rows, bool)
    named[order[outside]] = False
    order[outside] = np.resize(np.array([-1, rows, 2 ** 31 - 1, -2 ** 31], np.int32), len(outside))
    grad, out = (rng.integers(-2, 3, size=(rows, channels)).astype(np.float32) for _ in range(2))
    want = np.where(named[:, None], np.where(out > 0, grad, np.float32(0)), np.float32(9.0))
    gate = np.zeros((rows, (channels + 63) // 64 * 64), bool)
    inside = (order >= 0) & (order < rows)
    gate[inside, :channels] = out[order[inside]] > 0
    gate[~inside] = True
    bits = np.packbits(gate, axis=1, bitorder="little").reshape(rows, -1, 8).transpose(1, 0, 2)
    d_grad, d_out, d_order = H.dev(H.to_storage(grad, dtype), dtype), H.dev(H.to_storage(out, dtype), dtype), H.dev(order, "i32")
    d_bits = tv.from_numpy(np.ascontiguousarray(bits)).cuda()
    need = int(lib.cumm_hip_column_sum_workspace(rows, channels))
    ws = tv.zeros([need], tv.uint8, 0)
    for source in ({"out": d_out.byte_pointer()}, {"gate": d_bits.byte_pointer()}):
        gated, sums = H.dev(H.to_storage(np.full_like(grad, 9.0), dtype), dtype), tv.zeros([channels], H.TV_DTYPE[dtype], 0)
        gs = _capi.GateSums(gated=gated.byte_pointer(), sums=sums.byte_pointer(), grad=d_grad.byte_pointer(), rows=rows, channels=channels,
                            workspace=ws.byte_pointer(), workspace_bytes=need, order=d_order.byte_pointer(), **source)
        _capi.check(lib.cumm_hip_gate_sums(ctypes.byref(gs), int(H.TV_DTYPE[dtype]), None))
        _capi.check(lib.cumm_hip_device_synchronize())
        np.testing.assert_array_equal(H.as_f32(H.host(gated), dtype), want)
        np.testing.assert_array_equal(H.host(sums).view(np.uint16), H.to_storage(want[named].sum(axis=0), dtype).view(np.uint16))


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_sums_of_no_rows_in_an_order(dtype):
    """No rows, nothing to gate, whatever order they would have: the sums are zeros."""
    lib, channels = _capi.lib(), 72
    sums, order, ws = H.dev(H.to_storage(np.full(channels, 3.0, np.float32), dtype), dtype), tv.zeros([64], tv.int32, 0), tv.zeros([4096], tv.uint8, 0)
    gs = _capi.GateSums(sums=sums.byte_pointer(), rows=0, channels=channels, workspace=ws.byte_pointer(), workspace_bytes=4096, order=order.byte_pointer())
    _capi.check(lib.cumm_hip_gate_sums(ctypes.byref(gs), int(H.TV_DTYPE[dtype]), None))
    _capi.check(lib.cumm_hip_device_synchronize())
    assert not H.host(sums).view(np.uint16).any()


@pytest.mark.parametrize("cin,k_out", [(64, 64), (520, 64), (64, 136)])      # (a contraction of 520: the gate is a launch of its own)
def test_a_gate_of_positions_that_name_no_row(cin, k_out):
    """The bits of those positions are left alone, the others are what they are."""
    print("case gate of no row", cin, k_out, flush=True)
    rng, n = np.random.default_rng(cin + k_out), 300
    p = ConvParams(3, ConvOpType.Forward)
    p.conv_algo_desp = H.find_conv_desp("f16", ConvOpType.Forward, 64, 64)
    order = rng.permutation(n).astype(np.int32)
    inside = np.ones(n, bool)
    inside[[0, 7, 128, 299]] = False
    order[~inside] = [-1, n, 2 ** 31 - 1, -2 ** 31]
    p.input = H.dev(H.to_storage(rng.normal(0, 1, size=(n, cin)).astype(np.float32), "f16"), "f16")
    p.weight = H.dev(H.to_storage(rng.normal(0, 0.05, size=(k_out, 1, cin)).astype(np.float32), "f16"), "f16")
    p.output, p.act_type = tv.zeros([n, k_out], tv.float16, 0), Activation.ReLU
    p.indices, p.mask, p.mask_argsort = H.dev(np.arange(n, dtype=np.int32)[None], "i32"), H.dev(np.ones(n, np.uint32), "u32"), H.dev(order, "i32")
    ConvMainUnitTest.implicit_gemm2(p)
    groups = (k_out + 63) // 64
    d_gate = tv.from_numpy(np.full((groups, n, 8), 0xA5, np.uint8)).cuda()
    _again(p, gate=d_gate.byte_pointer())
    got = H.host(d_gate).transpose(1, 0, 2).reshape(n, groups * 8)[:, :k_out // 8]
    out = H.as_f32(H.host(p.output), "f16")
    np.testing.assert_array_equal(got[inside], np.packbits(out[order[inside]] > 0, axis=1, bitorder="little"))
    assert (got[~inside] == 0xA5).all()


def test_a_gate_has_a_position_for_every_row():
    """The bits of a call with another number of positions are not those of the rows."""
    n = 64
    p = ConvParams(3, ConvOpType.BackwardWeight)
    p.conv_algo_desp = H.find_conv_desp("f16", ConvOpType.BackwardWeight, 64, 64, split_k_parallel=True)
    p.input, p.output, p.weight = (tv.zeros(shape, tv.float16, 0) for shape in ([n, 64], [n, 64], [64, 1, 64]))
    p.indices, p.mask, p.mask_argsort = (H.dev(np.arange(n, dtype=np.int32)[None], "i32"), H.dev(np.ones(1, np.uint32), "u32"),
                                         H.dev(np.arange(n, dtype=np.int32), "i32"))
    p.mask_width, p.split_k_slices = 64, 4
    ConvMainUnitTest.implicit_gemm2(p)
    ws, gate, grad = (tv.zeros([1 << 16], tv.uint8, 0) for _ in range(3))
    gs = _capi.GateSums(gated=p.output.byte_pointer(), sums=ws.byte_pointer(), grad=grad.byte_pointer(), rows=n, channels=64,
                        workspace=ws.byte_pointer() + 4096, workspace_bytes=1 << 15, gate=gate.byte_pointer(), order=p.mask_argsort.byte_pointer())
    _again(p, sums=ctypes.addressof(gs))
    p.__dict__["_prepared"][5].N = n - 1
    with pytest.raises(ValueError):
        _again(p, sums=ctypes.addressof(gs))


@pytest.mark.parametrize("source", ["rows", "bias"])
@pytest.mark.parametrize("n", [60000, 9000])      # (one group of waves per tile, and two)
def test_f16_sums_with_a_source_round_alike_in_every_tile(source, n):
    """alpha * x + a source without an activation, x an exact sum: every result is one rounding of the exact value or
    of its fp32 rounding - the compiler takes some conversions into the fma - and the same bits whatever the tile."""
    print("case rounding with a source", source, n, flush=True)
    rng, c, alpha = np.random.default_rng(1), 64, 0.33371234
    x, src = (rng.normal(0, 1, size=(n, c)).astype(np.float16) for _ in range(2))
    if source == "bias":
        src = np.repeat(src[:1], n, axis=0)
    exact = np.float64(np.float32(alpha)) * x + src.astype(np.float64)      # (24 + 11 bits, and 11)
    one, two = exact.astype(np.float16), exact.astype(np.float32).astype(np.float16)
    assert (one != two).sum() > 20
    w = np.zeros((c, 1, c), np.float16)
    w[np.arange(c), 0, np.arange(c)] = 1
    rows, first = np.arange(n, dtype=np.int32), None
    for tile in ((64, 64), (128, 64), (64, 128), (128, 128)):
        p = ConvParams(3, ConvOpType.Forward)
        p.conv_algo_desp = H.find_conv_desp("f16", ConvOpType.Forward, *tile)
        p.input, p.output, p.weight = H.dev(x, "f16"), H.dev(src, "f16"), H.dev(w, "f16")
        p.indices, p.mask, p.mask_argsort = H.dev(rows[None], "i32"), H.dev(np.ones(n, np.uint32), "u32"), H.dev(rows, "i32")
        p.alpha, p.beta = alpha, 1.0
        if source == "bias":
            p.bias = H.dev(np.ascontiguousarray(src[0]), "f16")
        for hint in (0, -1):      # (mixed tile shapes, and one)
            p.light_prefix = hint
            if source == "rows":
                p.output = H.dev(src, "f16")
            ConvMainUnitTest.implicit_gemm2(p)
            got = H.host(p.output).view(np.uint16)
            assert ((got == one.view(np.uint16)) | (got == two.view(np.uint16))).all()
            first = got if first is None else first
            np.testing.assert_array_equal(got, first)


@pytest.mark.parametrize("ksize,channels,k_out,tile,hint", [
    (5, 64, 64, (64, 64), 0), (5, 136, 40, (128, 128), 0),                       # several mask words
    (3, 64, 520, (64, 64), 0), (3, 64, 520, (128, 128), 0), (3, 72, 264, (64, 128), -1)])      # kernels whose waits the compiler counts; chunks
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_write_empty_in_every_kernel(dtype, ksize, channels, k_out, tile, hint):
    """As test_write_empty, in the kernels of several mask words and of long contractions."""
    print("case write empty", dtype, ksize, channels, k_out, tile, hint, flush=True)
    rng, grid = np.random.default_rng(12), (12, 40, 36)
    coords = synth.clustered_voxels(rng, 1500, grid, 6, sigma=3.0)
    zz, yy = np.meshgrid(np.arange(grid[0]), np.arange(grid[1]), indexing="ij")
    planes = [np.stack([np.zeros(zz.size, np.int64), zz.ravel(), yy.ravel(), np.full(zz.size, grid[2] - 1)], axis=1)]
    coords = np.unique(np.concatenate([coords] + planes).astype(np.int32), axis=0)
    # (a padding that leaves the last plane without an output)
    pt = pairs.sparse_conv_pairs(coords, grid, ksize=(ksize,) * 3, padding=(0, 0, 0))
    n_in, n_out, kv = coords.shape[0], pt.indices_fwd.shape[1], ksize ** 3
    mask = pairs.masks_from_pairs(pt.indices_bwd)
    none = (mask == 0).all(axis=1)
    assert none.sum() >= 300
    w = H.to_storage(rng.normal(0, 0.05, size=(k_out, kv, channels)).astype(np.float32), dtype)
    dout = H.to_storage(rng.normal(0, 1, size=(n_out, k_out)).astype(np.float32), dtype)
    p = ConvParams(3, ConvOpType.BackwardInput)
    p.conv_algo_desp = H.find_conv_desp(dtype, ConvOpType.BackwardInput, *tile, dynamic_mask=kv > 32)
    p.input = H.dev(H.to_storage(np.full((n_in, channels), 7.0, np.float32), dtype), dtype)
    p.weight, p.output, p.indices = H.dev(w, dtype), H.dev(dout, dtype), H.dev(pt.indices_bwd, "i32")
    if kv > 32:
        p.mask, p.mask_argsort = pairs.sort_by_mask_words_device(H.dev(mask, "u32"))
        p.mask_int_count = mask.shape[1]
    else:
        ms, order = pairs.sort_by_mask(mask[:, 0])
        p.mask, p.mask_argsort = H.dev(ms, "u32"), H.dev(order, "i32")
        p.light_prefix = hint
    ConvMainUnitTest.implicit_gemm2(p)
    base = H.as_f32(H.host(p.input), dtype)
    assert (base[none] == 7.0).any()
    _again(p, write_empty=1)
    got = H.as_f32(H.host(p.input), dtype)
    assert (got[none] == 0.0).all()
    np.testing.assert_array_equal(got[~none], base[~none])
