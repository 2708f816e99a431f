"""The kernels with 256 x 256 tiles at the edges of their tiles, slabs and epilogues.  At these sizes quant_dot leaves
most calls to the register-staged kernel, so the tests that describe the large tiles run here with the
kernel named."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests import test_gpu_quant_dot as base
from tests.gpu_util import dev
from tests.quant_dot_kernel import Forced

pytestmark = pytest.mark.gpu


def _forced(monkeypatch, kernel):
    from amdmigraphx_amd import ops
    handle = Forced(kernel)
    monkeypatch.setattr(ops, "lib", lambda: handle)
    yield ops
    assert handle.taken > 0, "no call of this test is one for the kernel"


class TestDirectToLds:
    """one pass, K in shares with atomic adds (bare int8), four and eight waves"""

    @pytest.fixture
    def ops(self, monkeypatch):
        yield from _forced(monkeypatch, "dma")

    test_skinny_batched = staticmethod(base.test_int8_skinny_batched)
    test_extremes = staticmethod(base.test_int8_extremes_and_batch)
    test_epilogue = staticmethod(base.test_int8_dequant_epilogue_bit_exact)
    test_fp8_epilogue = staticmethod(base.test_fp8_dequant_epilogue)
    test_fp8_small_integers = staticmethod(base.test_fp8_small_integers_are_exact)
    test_fp8_four_wave_accumulators = staticmethod(base.test_fp8_four_wave_kernel_accumulators)

    # B as [K, N] is a call for these kernels where N is a multiple of 16, so the sizes beside those of the
    # tests that run here are theirs with the next such N

    @pytest.mark.parametrize("m,n,k", [(16, 8192, 8192), (128, 2048, 4096), (1, 256, 2048), (37, 512, 1088),
                                       (300, 272, 1024), (1024, 1024, 1024), (16, 768, 576)])
    @pytest.mark.parametrize("trans_b", [False, True])
    def test_skinny(self, ops, m, n, k, trans_b):
        base.test_int8_skinny_split_k_bit_exact(ops, m, n, k, trans_b)

    # K in shares through a workspace
    @pytest.mark.parametrize("m,n,k,batch,trans_b", [
        (16, 1024, 4096, 1, False), (128, 512, 2048, 1, False), (1, 256, 8192, 1, True), (33, 260, 1024, 2, True),
        (8, 256, 2112, 1, False), (16, 1023, 4096, 1, True), (40, 301, 1600, 2, True)])
    def test_shares(self, ops, m, n, k, batch, trans_b):
        base.test_int8_split_k_with_workspace_bit_exact(ops, m, n, k, batch, trans_b)

    @pytest.mark.parametrize("m,n,k,trans_b", [(16, 1024, 4096, False), (128, 768, 3072, True), (40, 304, 1600, False),
                                               (1, 512, 8192, True), (24, 250, 2048, True), (17, 49, 4608, True)])
    @pytest.mark.parametrize("out", ["f32", "f16", "bf16"])
    def test_shares_epilogue(self, ops, m, n, k, trans_b, out):
        base.test_int8_split_k_with_workspace_dequantizing_epilogue(ops, m, n, k, trans_b, out)

    test_fp8_shares = staticmethod(base.test_fp8_split_k_with_workspace)

    @pytest.mark.parametrize("m,n,k,batch,trans_b", [(300, 528, 3136, 32, False), (300, 520, 3136, 32, True),
                                                     (256, 512, 3072, 64, False), (513, 260, 3200, 24, True)])
    def test_four_wave_bare(self, ops, m, n, k, batch, trans_b):
        base.test_four_wave_kernel_bare_bit_exact(ops, m, n, k, batch, trans_b)

    @pytest.mark.parametrize("k", [3392, 3456, 3776, 3840, 4160, 7744])
    @pytest.mark.parametrize("trans_b,n", [(False, 528), (True, 520)])
    def test_four_wave_trips(self, ops, k, trans_b, n):
        base.test_four_wave_kernels_trip_boundaries_bit_exact(ops, k, trans_b, n)

    @pytest.mark.parametrize("m,n,k,trans_b", [(260, 272, 3072, False), (512, 520, 3136, True), (100, 1040, 4160, False)])
    @pytest.mark.parametrize("zp_a,zp_b", [(0, 0), (7, -9)])
    @pytest.mark.parametrize("out", ["f32", "f16", "bf16"])
    def test_four_wave_epilogue(self, ops, m, n, k, trans_b, zp_a, zp_b, out):
        base.test_four_wave_kernel_dequantizing_epilogue_bit_exact(ops, m, n, k, trans_b, zp_a, zp_b, out)

    @pytest.mark.parametrize("fp8", [False, True])
    def test_four_wave_unaligned_columns(self, ops, fp8):
        base.test_four_wave_kernel_unaligned_column_arrays(ops, fp8, 272)

    @pytest.mark.parametrize("k", [1024, 3072])
    @pytest.mark.parametrize("fp8", [False, True])
    @pytest.mark.parametrize("out", ["bare", "f32", "bf16"])
    def test_strided_views(self, ops, k, fp8, out):
        base.test_results_through_the_lds_copy_into_strided_batched_views(ops, k, fp8, out, 272)

    def test_four_wave_row_scales(self, ops):
        base.test_four_wave_kernel_per_row_scales(ops, 272)

    @pytest.mark.parametrize("m,n,k,batch,trans_b", [
        (260, 272, 3072, 1, False), (512, 520, 3200, 1, True), (100, 1040, 4224, 1, False),
        (256, 256, 3072, 2, True), (1024, 768, 3968, 1, False)])
    def test_fp8_four_wave_exact(self, ops, m, n, k, batch, trans_b):
        base.test_fp8_four_wave_kernel_small_integers_exact(ops, m, n, k, batch, trans_b)

    @pytest.mark.parametrize("m,n,k,trans_b", [(260, 272, 3072, False), (512, 520, 3200, True), (100, 1028, 4224, True),
                                               (77, 130, 3072, True)])
    @pytest.mark.parametrize("out", ["f32", "f16", "bf16"])
    @pytest.mark.parametrize("row_scales", [False, True])
    def test_fp8_four_wave_epilogue(self, ops, m, n, k, trans_b, out, row_scales):
        base.test_fp8_four_wave_kernel_dequantizing_epilogue(ops, m, n, k, trans_b, out, row_scales)

    @pytest.mark.parametrize("m,n,k,trans_b", [(192, 320, 2048, False), (512, 768, 768, True), (100, 272, 128, False),
                                               (64, 132, 256, True), (300, 1008, 512, False)])
    @pytest.mark.parametrize("out", ["f32", "f16", "bf16"])
    def test_bias(self, ops, m, n, k, trans_b, out):
        base.test_int8_bias_epilogue_bit_exact(ops, m, n, k, trans_b, out)

    @pytest.mark.parametrize("m,n", [(200, 272), (77, 512), (130, 1008)])
    @pytest.mark.parametrize("out", ["f16", "bf16"])
    def test_fp8_16bit_outputs(self, ops, m, n, out):
        base.test_fp8_16bit_outputs_ragged_shapes(ops, m, n, out)


class TestRegisterStagedLargeTiles:
    """csrc/qgemm_mfma.hip, K that is no multiple of 64"""

    @pytest.fixture
    def ops(self, monkeypatch):
        yield from _forced(monkeypatch, "mfma")

    # one slab of 128 and less, several and a remainder, ragged M and N
    SHAPES = [(1, 4, 16), (300, 260, 144), (257, 516, 272), (513, 132, 784), (255, 1028, 48)]

    @pytest.mark.parametrize("m,n,k", SHAPES)
    @pytest.mark.parametrize("trans_b", [False, True])
    def test_int8_sums(self, ops, m, n, k, trans_b):
        base.test_int8_accumulators_bit_exact(ops, m, n, k, trans_b)

    @pytest.mark.parametrize("m,n,k", SHAPES[1:])
    @pytest.mark.parametrize("trans_b", [False, True])
    @pytest.mark.parametrize("out", ["f32", "f16", "bf16"])
    def test_int8_epilogue(self, ops, m, n, k, trans_b, out):
        """a bias, and with odd M the zero point of A"""
        base.test_int8_bias_epilogue_bit_exact(ops, m, n, k, trans_b, out)

    @pytest.mark.parametrize("m,n,k", SHAPES)
    @pytest.mark.parametrize("trans_b", [False, True])
    def test_fp8_small_integers(self, ops, m, n, k, trans_b):
        rng = np.random.default_rng(m + n + k)
        a = orc.fp8_from_f32(rng.integers(-8, 9, (m, k)).astype(np.float32))
        b = orc.fp8_from_f32(rng.integers(-8, 9, (k, n)).astype(np.float32))
        db = dev(np.ascontiguousarray(b.T)).t() if trans_b else dev(b)
        want = orc.quant_dot(a, b, orc.FP8)
        assert np.array_equal(ops.quant_dot(dev(a), db, fp8=True).cpu().numpy(), want)
        # row and column scales and a bias behind exact sums
        sa, sb = (rng.uniform(0.01, 0.05, s).astype(np.float32) for s in (m, n))
        bias = rng.standard_normal(n).astype(np.float32)
        v = (want.astype(np.float64) * (sa[:, None] * sb[None]).astype(np.float64)).astype(np.float32) + bias
        got = ops.quant_dot(dev(a), db, fp8=True, scale_a=dev(sa), scale_b=dev(sb), bias=dev(bias),
                            out_dtype=torch.float32)
        assert np.array_equal(got.cpu().numpy().view(np.uint32), v.view(np.uint32))
