"""quant_dot's choice of a kernel, asked on the host (no GPU)."""
import os

import pytest

from amdmigraphx_amd import capi
from tests.quant_dot_kernel import kernel_of, small_shares

pytestmark = pytest.mark.skipif(not os.path.exists(capi.lib_path()), reason="library not built in this checkout")


def test_register_staged_kernel_keeps_room_for_its_read_ahead():
    """It counts K in ints and asks for positions up to two slabs of 256 and 240 bytes behind the last slab: with
    K up to 767 short of 2^31 such a position would wrap around to an address far in front of the matrix."""
    for k in (2**31 - 256, 2**31 - 257, 2**31 - 767, 2**31 - 1023, 2**31 - 1024):
        assert kernel_of(1, 1, k, trans_b=True) == "generic"
    last = 2**31 - 1025
    furthest = ((last + 255) // 256 + 1) * 256 + 240
    assert furthest < 2**31
    assert kernel_of(1, 1, last, trans_b=True) == "ragged_exact"


def test_register_staged_kernel_keeps_to_the_largest_grid():
    """2^24 workgroups of 256 threads are more than one launch takes; 180 GB of bfloat16 results still fit the card."""
    m = 300001
    assert (m + 63) // 64 * ((m + 63) // 64) * 256 >= 2**32
    assert kernel_of(m, m, 17, fp8=True, out="bf16") == "generic"
    assert kernel_of(250001, 250001, 17, fp8=True, out="bf16") == "ragged_exact"
    assert (m + 127) // 128 * ((m + 127) // 128) * 256 < 2**32
    assert kernel_of(m, m, 17, out="bf16") == "ragged_exact"


@pytest.mark.parametrize("m,n,k,trans_b,kernel", [
    # bare int8 without a workspace: few tiles of a long K are split over the chip with atomic adds ...
    (16, 8192, 8192, False, "dma_atomic"), (16, 2048, 8192, True, "dma_atomic"), (16, 256, 25600, False, "dma_atomic"),
    (16, 256, 25600, True, "dma_atomic"), (1, 64, 26688, True, "dma_atomic"), (5, 192, 25472, False, "dma_atomic"),
    (264, 128, 19968, False, "dma_atomic"),
    # ... but not where the adds or the long way of B cost more than they gain, or K is short
    (16, 8192, 8192, True, "ragged"), (128, 8192, 8192, False, "ragged"), (128, 8192, 8192, True, "ragged"),
    (16, 1024, 1024, False, "ragged"), (256, 512, 2048, True, "ragged")])
def test_bare_int8_product_is_compared_with_the_split_it_would_run(m, n, k, trans_b, kernel):
    """Measured, split against register-staged: 5 x 192 x 25472 16.4 / 79.9 us, 16 x 8192 x 8192 30.1 / 36.7 and with B
    as [N, K] 30.7 / 23.6, 128 x 8192 x 8192 71.0 / 39.3 and 74.6 / 26.0."""
    assert kernel_of(m, n, k, trans_b=trans_b) == kernel


@pytest.mark.parametrize("m,n,k,trans_b,kernel", [
    (16, 8192, 8192, False, "dma_shares"), (128, 8192, 8192, False, "dma_shares"), (16, 2048, 8192, True, "dma_shares"),
    (128, 14336, 4096, False, "dma_shares"), (128, 8192, 8192, True, "ragged"), (512, 2048, 8192, True, "ragged"),
    (512, 4096, 4096, False, "ragged"), (512, 4096, 4096, True, "ragged")])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("out", [None, "bf16"])
def test_a_workspace_is_used_where_the_shares_are_faster(m, n, k, trans_b, kernel, fp8, out):
    """Measured, shares against register-staged: 128 x 8192 x 8192 fp8 34.5 / 39.3 us, with B as [N, K] 34.5 / 25.3;
    512 x 4096 x 4096 33.5 / 28.0."""
    assert kernel_of(m, n, k, trans_b=trans_b, fp8=fp8, out=out, workspace=64 << 20) == kernel
    # one that is too small is none
    assert kernel_of(m, n, k, trans_b=trans_b, fp8=fp8, out=out, workspace=1 << 10) in ("ragged", "dma_atomic")


@pytest.mark.parametrize("m,n,k,trans_b,fp8", [
    (640, 1520, 6656, False, True), (897, 400, 6016, False, True), (142, 2128, 5504, False, True),
    (543, 1376, 4224, False, False), (291, 912, 2752, False, False), (127, 6304, 3776, False, False),
    (16, 512, 4096, False, True), (16, 512, 4096, False, False), (1, 16, 4160, True, True), (1, 16, 4160, True, False)])
def test_the_size_asked_for_serves_any_distance_of_the_rows(m, n, k, trans_b, fp8):
    """rows of B that lie a multiple of 1 KiB apart take another time, yet the size is asked for without it"""
    from amdmigraphx_amd import ops
    need = ops.quant_dot_workspace_size(m, n, k, trans_b=trans_b, fp8=fp8)
    kernel = kernel_of(m, n, k, trans_b=trans_b, fp8=fp8, workspace=need)
    for ldb in ((k if trans_b else n) + 1023) // 1024 * 1024, ((k if trans_b else n) + 1039) // 16 * 16:
        for lda in (k, k + 64):
            assert kernel_of(m, n, k, trans_b=trans_b, fp8=fp8, lda=lda, ldb=ldb, workspace=need) == kernel


@pytest.mark.parametrize("m,n,k", [(128, 4096, 8128), (128, 4096, 14272), (64, 4096, 4288), (128, 2048, 8128), (344, 400, 6016)])
def test_fp8_shares_need_no_divisor_of_k(m, n, k):
    """slabs of K are dealt to the shares in small tiles, whose last one may be the shorter, for either type"""
    assert small_shares(m, n, k, fp8=True) == small_shares(m, n, k) > 1


@pytest.mark.parametrize("m,n,k", [(64, 256, 2112), (606, 288, 4160), (128, 4096, 8192)])
def test_fp8_shares_are_equal_where_that_costs_little(m, n, k):
    from amdmigraphx_amd import ops
    shares = ops.quant_dot_workspace_size(m, n, k, fp8=True) // (4 * m * n)
    assert shares > 1 and shares != small_shares(m, n, k) and k // 64 % shares == 0


@pytest.mark.parametrize("m,n,k,trans_b,fp8", [(318, 1664, 12672, True, False), (750, 880, 12480, True, True),
                                               (255, 8192, 8192, False, False)])
def test_the_static_entry_refuses_by_the_large_tiles(m, n, k, trans_b, fp8):
    """two products that would split in small tiles with less than the buffer, and one that would not"""
    import ctypes
    from amdmigraphx_amd import ops
    d = capi.QuantDotDesc(m=m, n=n, k=k, lda=k, ldb=k if trans_b else n, ldc=n, batch=1, trans_b=int(trans_b),
                          in_type=capi.DT.FP8 if fp8 else capi.DT.I8, out_type=capi.DT.F32 if fp8 else capi.DT.I32)
    status = capi.lib().mi355_quant_dot_static(ctypes.byref(d), *[ctypes.c_void_p(1 << 20)] * 3, *[None] * 6)
    assert status == -4  # MI355_ERR_SCRATCH_TOO_SMALL
    assert (ops.quant_dot_workspace_size(m, n, k, trans_b=trans_b, fp8=fp8) > 32 << 20) == (m == 255)


@pytest.mark.parametrize("batch,m,n,k,fp8,out", [
    (1, 10, 58608, 128, False, None), (1, 1, 2896, 16, True, None), (1, 8, 4996, 32, True, None), (3, 26, 16, 16, True, None),
    (1, 2, 23956, 32, True, "f32"), (18, 282, 16, 64, True, None), (1, 26278, 16, 64, True, None), (477, 18, 236, 32, True, "f32")])
def test_one_slab_of_few_rows(batch, m, n, k, fp8, out):
    """Measured, one slab against the kernel of 256 x 256 tiles that a fit without the small start of bare results had
    chosen: 3.7 / 7.4 us, 2.8 / 5.1, 3.0 / 5.3, 3.0 / 5.0, 3.4 / 5.7, 3.3 / 4.8, 3.6 / 5.0, 8.0 / 12.4."""
    assert kernel_of(m, n, k, trans_b=True, fp8=fp8, out=out, batch=batch) == "ragged"


@pytest.mark.parametrize("batch,m,n,k,out", [(14, 882, 882, 64, "f32"), (1, 3058, 38471, 64, "bf16"), (1, 7187, 24363, 64, None),
                                             (451, 963, 527, 128, "bf16"), (1, 4447, 29009, 64, None)])
@pytest.mark.parametrize("fp8", [False, True])
def test_rows_that_are_no_whole_groups_of_4(batch, m, n, k, out, fp8):
    """Short K: the large tiles store such rows element by element (46 us against 12, 328 / 105, 519 / 254, 654 / 245,
    398 / 174)"""
    assert kernel_of(m, n, k, trans_b=True, fp8=fp8, out=out, batch=batch) == "ragged"


def test_large_and_small_grids():
    for fp8 in (False, True):
        for out in (None, "bf16", "f32"):
            assert kernel_of(8192, 8192, 8192, fp8=fp8, out=out) == "dma"
            assert kernel_of(4096, 4096, 4096, fp8=fp8, out=out) == "dma"
            assert kernel_of(1024, 1024, 1024, fp8=fp8, out=out) == "ragged"
            assert kernel_of(4096, 4096, 4112, fp8=fp8, out=out) == "mfma"
            assert kernel_of(197, 64, 208, batch=96, fp8=fp8, out=out) == "ragged"
    # a vector of column scales per batch entry: only the direct-to-LDS kernels have it
    assert kernel_of(128, 768, 768, batch=3, out="f32", scale_b_mode=capi.QP.PER_COL_BATCH) == "dma"


@pytest.mark.parametrize("m,n,k,batch,kernel", [
    (44, 87, 17, 1, "generic"), (356, 45, 17, 1, "generic"), (1, 5, 16, 1, "generic"), (74, 7, 31, 1, "generic"),
    # many outputs, or more of K than a few blocks are done with at once
    (2049, 2051, 17, 1, "ragged_exact"), (33, 35, 17, 500, "ragged_exact"), (65, 63, 93, 1, "ragged_exact"),
    (500, 30522, 768, 1, "ragged_exact"), (197, 197, 61, 96, "ragged_exact")])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("out", [None, "bf16"])
def test_short_unaligned_k(m, n, k, batch, kernel, fp8, out):
    assert kernel_of(m, n, k, batch=batch, fp8=fp8, out=out) == kernel
