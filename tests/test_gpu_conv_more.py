"""cumm_hip_sparse_conv_more: what a training program wants of the convolution launches beyond the reference's
argument block."""
import ctypes

import numpy as np
import pytest

import helpers as H
from cumm_amd import _capi, pairs, synth
from cumm_amd.conv.main import ConvMainUnitTest
from cumm_amd.tensorview.gemm import ConvOpType, ConvParams

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
