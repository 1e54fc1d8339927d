"""The kernels that launches of many tiles take - tiles of two shapes in one launch (the light end in pairs, the heavy
end in halves), contractions of several steps, several mask words - at the sizes of the cases that the oracle
checks.  Those cases are launches of few tiles, whose 64 x 64 tiles go to two groups of waves; with
``deterministic`` they do not, and hints move work between the kernels of one order of the sums."""
import pytest

import test_gpu_conv as conv
import test_gpu_random_dynamic as random_dynamic
import test_gpu_random_shapes as random_shapes
from cumm_amd.conv.main import ConvMainUnitTest
from cumm_amd.tensorview.gemm import ConvOpType

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def one_order(monkeypatch):
    call = ConvMainUnitTest.implicit_gemm2

    def in_one_order(p):
        if ConvOpType(p.conv_algo_desp.op_type) != ConvOpType.BackwardWeight:
            p.deterministic = True
        call(p)
    monkeypatch.setattr(ConvMainUnitTest, "implicit_gemm2", staticmethod(in_one_order))


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("c_in,k_out", [(64, 64), (32, 48), (16, 24)])
def test_hints_of_every_size(dtype, c_in, k_out):
    conv.test_light_prefix_hint_moves_work_not_results(dtype, c_in, k_out)


def test_halves_of_a_pair_without_any_offset():
    conv.test_light_prefix_leaves_skipped_rows_alone()


def test_ragged_sizes_and_hints_past_the_end():
    conv.test_ragged_and_empty()


@pytest.mark.parametrize("dtype,c_in,k_out", [("f16", 64, 64), ("bf16", 64, 64), ("bf16", 48, 40), ("f16", 32, 32), ("bf16", 32, 24)])
@pytest.mark.parametrize("n_target", [12000, 2100])
def test_pairs_and_halves(dtype, c_in, k_out, n_target):
    conv.test_order_by_offset_count_and_half_tiles(dtype, c_in, k_out, n_target)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("c_in,k_out", [(128, 128), (72, 40), (200, 64)])
def test_contractions_of_several_steps(dtype, c_in, k_out):
    conv.test_subm_forward(dtype, (64, 64), c_in, k_out)


@pytest.mark.parametrize("block", range(3))
def test_random_shapes(block):
    random_shapes.test_random_shapes_against_the_oracle(block)


@pytest.mark.parametrize("block", range(2))
def test_random_kernel_volumes_above_32(block):
    random_dynamic.test_random_kernel_volumes_above_32(block)
