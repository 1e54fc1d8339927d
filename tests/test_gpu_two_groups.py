"""Launches of few 64 x 64 tiles, whose kernel offsets are shared by two groups of waves (launch_two_groups in
rowgemm_inst.hip): both sides of the line, one tile, offsets of one group only, contractions of one and of
several steps, against a float32 sum over the pair table; and rows whose bits do not depend on the order of
the positions."""
import pytest

import helpers as H
from cumm_amd import tensorview as tv
from cumm_amd.conv.main import ConvMainUnitTest
from cumm_amd.tensorview.gemm import ConvOpType, ConvParams

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# one rounding to the type, and fp32 sums of up to 125 x 136 products of values around 0.05
TOL = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}


def _words(table):
    kv, n = table.shape
    words = (kv + 31) // 32
    m = torch.zeros(n, words, dtype=torch.int64, device="cuda")
    for k in range(kv):
        m[:, k // 32] |= (table[k] >= 0).long() << (k % 32)
    m = torch.where(m >= 1 << 31, m - (1 << 32), m).to(torch.int32)
    return m if words > 1 else m[:, 0].contiguous()


def _run(op, dtype, table, x, w, order):
    from cumm_amd.torch_bridge import torch2tensor as t
    kv, n = table.shape
    mask = _words(table)
    p = ConvParams(3, op)
    p.conv_algo_desp = H.find_conv_desp(dtype, op, 64, 64, dynamic_mask=kv > 32)
    out = torch.full((n, w.shape[0] if op == ConvOpType.Forward else w.shape[2]), 7.0, dtype=x.dtype, device="cuda")
    if op == ConvOpType.Forward:
        p.input, p.output = t(x), t(out)
    else:
        p.output, p.input = t(x), t(out)
    p.weight, p.indices = t(w), t(table)
    sorted_mask = mask[order.long()].contiguous()
    p.mask = tv.from_blob_strided(sorted_mask.data_ptr(), [n] if kv <= 32 else [n, mask.shape[1]],
                                  [1] if kv <= 32 else [mask.shape[1], 1], tv.uint32, 0, keepalive=sorted_mask)
    p.mask_argsort = t(order)
    p.mask_int_count = (kv + 31) // 32
    ConvMainUnitTest.implicit_gemm2(p)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("op", [ConvOpType.Forward, ConvOpType.BackwardInput])
@pytest.mark.parametrize("dtype,kv,c,k,n,which", [
    ("f16", 27, 64, 64, 1, "all"), ("f16", 27, 64, 64, 63, "centre"), ("bf16", 27, 16, 24, 65, "all"),
    ("f16", 27, 64, 64, 64 * 384, "all"), ("f16", 27, 64, 64, 64 * 384 + 1, "all"),
    ("bf16", 27, 32, 64, 64 * 1024, "all"), ("bf16", 27, 32, 64, 64 * 1024 + 1, "all"),
    ("f16", 27, 136, 128, 64 * 512 + 1, "all"),
    ("f16", 27, 136, 128, 64 * 512, "all"), ("f16", 27, 128, 72, 4000, "even"),
    ("f16", 32, 64, 64, 500, "all"), ("bf16", 9, 48, 64, 700, "all"), ("f16", 1, 64, 64, 200, "all"),
    ("f16", 125, 64, 64, 1000, "all"), ("bf16", 125, 24, 64, 64, "centre"), ("f16", 75, 72, 64, 300, "all"),
    ("bf16", 125, 64, 64, 64 * 1024 + 1, "even")])
def test_against_the_sum_over_the_table(op, dtype, kv, c, k, n, which):
    print("case two groups", op, dtype, kv, c, k, n, which, flush=True)
    torch.backends.cuda.matmul.allow_tf32 = False
    gen = torch.Generator(device="cuda").manual_seed(kv * 1000 + n)
    tdt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    rows = n + 5
    table = torch.randint(0, rows, (kv, n), generator=gen, device="cuda", dtype=torch.int32)
    keep = torch.rand(kv, n, generator=gen, device="cuda") < (0.3 if n < 5000 else 4.0 / kv)
    if which == "centre":
        keep[:] = False
        keep[kv // 2] = True
    elif which == "even":
        keep[1::2] = False
    table = torch.where(keep, table, -1).contiguous()
    contraction = c if op == ConvOpType.Forward else k
    x = torch.randn(rows, contraction, generator=gen, device="cuda").to(tdt)
    w = (torch.randn(k, kv, c, generator=gen, device="cuda") * 0.05).to(tdt)
    order = torch.argsort(_words(table) if kv <= 32 else _words(table)[:, 0], stable=True).to(torch.int32)
    got = _run(op, dtype, table, x, w, order)
    ref = torch.zeros(n, k if op == ConvOpType.Forward else c, device="cuda")
    size = torch.zeros_like(ref)
    xf = torch.cat([x.float(), torch.zeros(1, contraction, device="cuda")])
    for i in range(kv):
        wk = w[:, i].float().t() if op == ConvOpType.Forward else w[:, i].float()
        a = xf[torch.where(table[i] >= 0, table[i], rows).long()]
        ref += a @ wk
        size += a.abs() @ wk.abs()
    if op == ConvOpType.BackwardInput:      # rows of tiles without any offset are left alone
        empty = (table < 0).all(0)[order.long()]
        pad = torch.ones((n + 63) // 64 * 64, dtype=torch.bool, device="cuda")
        pad[:n] = empty
        skipped = pad.view(-1, 64).all(1).repeat_interleave(64)[:n]
        ref[order.long()[skipped]] = 7.0
    bound = TOL[dtype] * ref.abs() + 2.0 ** -20 * size + 2.0 ** -24
    assert bool(((got.float() - ref).abs() <= bound).all())
    # any order of the positions: the same bits
    other = torch.randperm(n, generator=gen, device="cuda").to(torch.int32)
    again = _run(op, dtype, table, x, w, other)
    present = (table >= 0).any(0)
    assert torch.equal(got[present], again[present])


@pytest.mark.parametrize("op", [ConvOpType.Forward, ConvOpType.BackwardInput])
@pytest.mark.parametrize("dtype,kv,c,k", [("f16", 27, 64, 64), ("bf16", 27, 128, 136), ("f16", 27, 24, 32), ("bf16", 125, 64, 64)])
def test_one_order_on_request(monkeypatch, op, dtype, kv, c, k):
    """With ``deterministic`` a row has the same bits in every tile, and in a launch of 700 rows or of 70 000."""
    print("case one order", op, dtype, kv, c, k, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(kv + c)
    tdt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    rows, n, copies = 705, 700, 100
    table = torch.randint(0, rows, (kv, n), generator=gen, device="cuda", dtype=torch.int32)
    table = torch.where(torch.rand(kv, n, generator=gen, device="cuda") < 0.3, table, -1).contiguous()
    x = torch.randn(rows, c if op == ConvOpType.Forward else k, generator=gen, device="cuda").to(tdt)
    w = (torch.randn(k, kv, c, generator=gen, device="cuda") * 0.05).to(tdt)
    find, call = H.find_conv_desp, ConvMainUnitTest.implicit_gemm2

    def run(table, tile):
        order = torch.argsort(_words(table) if kv <= 32 else _words(table)[:, 0], stable=True).to(torch.int32)
        with monkeypatch.context() as m:
            m.setattr(H, "find_conv_desp", lambda *a, **k: find(*a[:2], tile, tile, **k))
            m.setattr(ConvMainUnitTest, "implicit_gemm2", staticmethod(lambda p: setattr(p, "deterministic", True) or call(p)))
            return _run(op, dtype, table, x, w, order)
    alone = [run(table, tile) for tile in (64, 128)]
    batch = [run(table.repeat(1, copies), tile).view(copies, n, -1) for tile in (64, 128)]
    present = (table >= 0).any(0)
    assert torch.equal(alone[0][present], alone[1][present])
    for b in batch:
        assert all(torch.equal(b[i][present], alone[0][present]) for i in range(copies))


@pytest.mark.parametrize("op", [ConvOpType.Forward, ConvOpType.BackwardInput])
@pytest.mark.parametrize("dtype,kv,c,k,n,which", [
    ("f16", 27, 136, 64, 64 * 384, "all"), ("f16", 27, 136, 64, 64 * 384 + 1, "all"), ("bf16", 32, 40, 72, 64 * 192, "all"),
    ("f16", 125, 32, 64, 64 * 512, "all"), ("bf16", 125, 64, 64, 64 * 512 + 1, "even"), ("bf16", 36, 16, 8, 1, "all"),
    ("bf16", 27, 136, 72, 64 * 128, "all"), ("f16", 27, 136, 64, 64 * 256, "even"), ("bf16", 27, 200, 64, 64 * 256 + 1, "all"),
    ("f16", 125, 64, 64, 64 * 256, "even"), ("bf16", 125, 32, 64, 64 * 256 + 1, "all")])
def test_sides_of_the_line_of_four_groups(op, dtype, kv, c, k, n, which):
    test_against_the_sum_over_the_table(op, dtype, kv, c, k, n, which)


@pytest.mark.parametrize("c_in,k_out", [(144, 64), (256, 48), (128, 64)])      # (several steps per offset: four groups; one: two)
def test_s8_of_few_tiles(c_in, k_out):
    import numpy as np
    from cumm_amd import pairs, synth
    from oracle import conv_ref
    print("case s8 of few tiles", c_in, k_out, flush=True)
    rng, grid = np.random.default_rng(c_in), (12, 40, 36)
    pt = pairs.subm_pairs(synth.clustered_voxels(rng, 3000, grid, 6, sigma=3.0), grid)
    n = pt.indices_fwd.shape[1]
    x, w = (rng.integers(-20, 21, size=s).astype(np.int8) for s in ((n, c_in), (k_out, 27, c_in)))
    scale, bias = rng.uniform(0.001, 0.01, size=k_out).astype(np.float32), rng.normal(0, 1, size=k_out).astype(np.float32)
    ms, order = pairs.sort_by_mask(pt.mask_fwd)
    out0 = np.zeros((n, k_out), np.int8)
    p = ConvParams(3, ConvOpType.Forward)
    p.conv_algo_desp = H.find_conv_desp("s8", ConvOpType.Forward, 64, 64, int8_inference=True)
    p.input, p.weight, p.output = H.dev(x, "s8"), H.dev(w, "s8"), H.dev(out0, "s8")
    p.scale, p.bias = H.dev(scale, "f32"), H.dev(bias, "f32")
    p.indices, p.mask, p.mask_argsort = H.dev(pt.indices_fwd, "i32"), H.dev(ms, "u32"), H.dev(order, "i32")
    ConvMainUnitTest.implicit_gemm2(p)
    ref, _ = conv_ref.implicit_gemm_fwd_ref(x, w, out0, pt.indices_fwd, ms, order, tile_m=64, dtype_in="s8", dtype_w="s8", dtype_out="s8",
                                            scale=scale, bias=bias, int8_inference=True)
    np.testing.assert_array_equal(H.host(p.output), ref)
