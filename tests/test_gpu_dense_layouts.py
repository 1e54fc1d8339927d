"""Dense matmul2 on the LDS-ring kernels in all layouts (densegemm_lds.h): tile edges and remainders in m, n
and k, each kernel of the dispatch, alpha / beta with a separate source and with a bias, against torch's
fp32 product of the same operands."""
import numpy as np
import pytest

import helpers as H
from cumm_amd import tensorview as tv
from cumm_amd.gemm.main import GemmMainUnitTest
from cumm_amd.tensorview.gemm import Activation, GemmParams, ShuffleStrideType

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# one rounding to the type of values around sqrt(k), and fp32 sums of k products
TOL = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}


def _run(dtype, m, n, k, ta, tb, source, alpha=1.0, beta=0.0, relu=False, tile=64):
    from cumm_amd.torch_bridge import torch2tensor
    tdt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    gen = torch.Generator(device="cuda").manual_seed(m * 131 + n * 17 + k)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(tdt)
    a, b = rnd(*((k, m) if ta else (m, k))), rnd(*((n, k) if tb else (k, n)))
    c = torch.full((m, n), float("nan"), dtype=tdt, device="cuda")
    p = GemmParams()
    p.algo_desp = H.find_gemm_desp(dtype, ShuffleStrideType.NoShuffle, tile, tile, ta, tb)
    p.a, p.b, p.c = torch2tensor(a), torch2tensor(b), torch2tensor(c)
    ref = alpha * ((a.float().t() if ta else a.float()) @ (b.float().t() if tb else b.float()))
    if source != "none":
        d = rnd(n) if source == "bias" else rnd(m, n)
        p.d = torch2tensor(d)
        ref = ref + beta * d.float()
    p.alpha, p.beta = alpha, beta
    if relu:
        p.act_type, ref = Activation.ReLU, ref.clamp_min(0)
    GemmMainUnitTest.matmul2(p)
    torch.cuda.synchronize()
    err = (c.float() - ref).abs()
    bound = TOL[dtype] * ref.abs() + 3e-6 * k ** 0.5 * 4 + 1e-6 + TOL[dtype] * 1e-2
    assert bool((err <= bound).all()), float((err - bound).max())


@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_edges_of_tiles_and_steps(dtype, ta, tb):
    torch.backends.cuda.matmul.allow_tf32 = False
    for m in (8, 64, 72, 200):
        for n in (8, 64, 136):
            for k in (8, 24, 32, 64, 72, 328):
                print("case dense", dtype, ta, tb, m, n, k, flush=True)
                _run(dtype, m, n, k, ta, tb, "none")
    # any number of rows of a row-major operand; any k where both operands have it as their row index
    if not ta:
        for m in (1, 63, 65, 191):
            _run(dtype, m, 72, 104, ta, tb, "none")
    if ta and not tb:
        for k in (1, 7, 33, 1001):
            _run(dtype, 72, 200, k, ta, tb, "none")


@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k", [(136, 72, 2056),        # k over eight waves
                                   (1000, 1064, 520),      # 64 x 64
                                   (1992, 2040, 1032),     # 128 x 64
                                   (2040, 2056, 1032),     # 128 x 128
                                   (4088, 4088, 1048)])    # 256 x 256
def test_each_kernel_with_its_epilogue(m, n, k, ta, tb):
    torch.backends.cuda.matmul.allow_tf32 = False
    print("case dense epilogue", m, n, k, ta, tb, flush=True)
    _run("f16", m, n, k, ta, tb, "matrix", alpha=0.5, beta=2.0)
    _run("bf16", m, n, k, ta, tb, "bias", alpha=1.0, beta=1.0, relu=True)


@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("tile", [64, 128])
def test_short_contractions_on_either_side_of_the_streaming_kernels(tile, ta, tb):
    """k from half a step to a step and a half, with fewer and with more than three tiles per CU, whatever tile
    the descriptor has: the register-staged kernel below the line, the streaming ones above it."""
    torch.backends.cuda.matmul.allow_tf32 = False
    for m, n in ((200, 136), (1992, 2056)):
        for k in (8, 32, 40, 64, 96, 104):
            print("case dense short", tile, m, n, k, ta, tb, flush=True)
            _run("f16", m, n, k, ta, tb, "matrix", alpha=0.5, beta=2.0, tile=tile)
            _run("bf16", m, n, k, ta, tb, "bias", alpha=1.0, beta=1.0, relu=True, tile=tile)


@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k", [(72, 136, 72),          # few tiles, one step and a remainder, two wave groups
                                   (72, 136, 1032),        # k over eight waves / 128 of k per step by the lines
                                   (1000, 1000, 136),      # 64 x 64, a tile per CU
                                   (1000, 1000, 904),      # 64 x 64, 128 of k per step, remainder of a group's slice
                                   (1992, 776, 1160),      # 64 x 128
                                   (2040, 1992, 1992),     # 128 x 128, a tile per CU
                                   (1992, 3336, 872)])     # 128 x 128, two tiles per CU
def test_kernels_of_eight_waves(m, n, k, ta, tb):
    """Every tile of the eight-wave kernels at ragged m, n and k: row and column remainders, a last step whose k
    ends inside one wave group's slice."""
    torch.backends.cuda.matmul.allow_tf32 = False
    print("case dense eight waves", m, n, k, ta, tb, flush=True)
    _run("f16", m, n, k, ta, tb, "matrix", alpha=0.5, beta=2.0)
    _run("bf16", m, n, k, ta, tb, "none")
