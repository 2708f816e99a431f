"""quant_dot of matrices aligned to nothing: the register-staged matrix-core kernel against the
oracle, bit for bit (int8: whole sums; fp8: digit sums put together in double, which is the
oracle's own double sum)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests.gpu_util import bf16_bits, dev, half_bits
from tests.quant_dot_kernel import kernel_of

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from amdmigraphx_amd import ops
    return ops


# edges of the 64 and 128 tiles and of the 64, 128 and 256 slabs, the smallest K and N taken, one
# short of a 16-byte piece and one beyond it
SHAPES = [(1, 4, 16), (64, 64, 64), (65, 63, 65), (63, 66, 127), (5, 129, 31), (130, 5, 257), (197, 64, 197),
          (197, 197, 61), (70, 1001, 250), (2049, 2051, 17), (2100, 2110, 143)]


def _fp8(rng, shape, nan):
    """every exponent, both zeros; without the NaN codes unless asked for"""
    v = rng.integers(0, 256, shape, dtype=np.uint8)
    return v if nan else np.where((v & 0x7f) == 0x7f, v - 1, v).astype(np.uint8)


def _on_device(x, trans, pad):
    """[K, N] as it lies, or as the transpose of [N, K]; rows `pad` elements longer than the matrix, which
    ends where its storage ends"""
    x = np.ascontiguousarray(x.T) if trans else x
    r, c = x.shape
    t = torch.full((r * (c + pad) - pad,), 0x7f, dtype=torch.uint8 if x.dtype == np.uint8 else torch.int8, device="cuda")
    t = torch.as_strided(t, (r, c), (c + pad, 1))
    t.copy_(dev(x))
    return t.t() if trans else t


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("fp8", [False, True])
def test_bare_sums(ops, m, n, k, trans_b, fp8):
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    if fp8:
        a, b = _fp8(rng, (m, k), False), _fp8(rng, (k, n), False)
        a[m // 2, k - 1] = 0x7f  # a NaN in the last piece of a row of A
        if n > 4:
            b[0, n - 1] = 0xff
    else:
        a, b = (rng.integers(-128, 128, s, dtype=np.int8) for s in ((m, k), (k, n)))
    want = orc.quant_dot(a, b, orc.FP8 if fp8 else orc.I8)
    # odd leading dimensions, so that no other kernel takes the call
    out = torch.full((m, n + 3), 7, dtype=torch.float32 if fp8 else torch.int32, device="cuda")
    print("ragged", m, n, k, trans_b, fp8, flush=True)
    ops.quant_dot(_on_device(a, False, 1), _on_device(b, trans_b, 3), fp8=fp8, out=out[:, :n])
    got = out.cpu().numpy()
    assert (got[:, n:] == 7).all()
    assert np.array_equal(got[:, :n], want.reshape(m, n), equal_nan=True)


@pytest.mark.parametrize("m,n,k", [(65, 63, 65), (197, 30, 197), (2100, 2110, 143)])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("out", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("zp_a,zp_b", [(0, 0), (7, -9)])
def test_int8_epilogue(ops, m, n, k, trans_b, out, zp_a, zp_b):
    rng = np.random.default_rng(m + n + k)
    a, b = (rng.integers(-128, 128, s, dtype=np.int8) for s in ((m, k), (k, n)))
    sa, sb = (rng.uniform(0.001, 0.01, s).astype(np.float32) for s in (m, n))
    bias = rng.standard_normal(n).astype(np.float32)
    acc = orc.quant_dot(a, b, orc.I8).reshape(m, n).astype(np.float64)
    zp = zp_a * b.astype(np.int64).sum(0)[None] + zp_b * a.astype(np.int64).sum(1)[:, None] - k * zp_a * zp_b
    v = ((acc - zp) * (sa[:, None] * sb[None]).astype(np.float64)).astype(np.float32) + bias
    odt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[out]
    da, db = _on_device(a, False, 1), _on_device(b, trans_b, 3)
    got = ops.quant_dot(da, db, scale_a=dev(sa), scale_b=dev(sb), zp_a=zp_a, zp_b=zp_b, bias=dev(bias),
                        colsum_b=dev(b.astype(np.int32).sum(0, dtype=np.int32)),
                        rowsum_a=dev(a.astype(np.int32).sum(1, dtype=np.int32)), out_dtype=odt)
    if out == "f32":
        assert np.array_equal(got.cpu().numpy().view(np.uint32), v.view(np.uint32))
    elif out == "f16":
        assert np.array_equal(half_bits(got), orc.convert(v, orc.F32, orc.F16).reshape(m, n))
    else:
        assert np.array_equal(bf16_bits(got), orc.convert(v, orc.F32, orc.BF16).reshape(m, n))


@pytest.mark.parametrize("trans_b", [False, True])
def test_fp8_epilogue_and_batches(ops, trans_b):
    rng = np.random.default_rng(5)
    nb, m, n, k = 3, 70, 67, 131
    a, b = _fp8(rng, (nb, m, k), False), _fp8(rng, (nb, k, n), False)
    sa, sb = (rng.uniform(0.001, 0.01, s).astype(np.float32) for s in (m, n))
    acc = np.stack([orc.quant_dot(a[i], b[i], orc.FP8).reshape(m, n) for i in range(nb)]).astype(np.float64)
    want = (acc * (sa[:, None] * sb[None]).astype(np.float64)).astype(np.float32)
    db = dev(np.ascontiguousarray(b.transpose(0, 2, 1))).transpose(1, 2) if trans_b else dev(b)
    got = ops.quant_dot(dev(a), db, fp8=True, scale_a=dev(sa), scale_b=dev(sb), out_dtype=torch.float32)
    assert np.array_equal(got.cpu().numpy().view(np.uint32), want.view(np.uint32))


def test_fp8_largest_digit_sums(ops):
    """the largest codes over the longest K the digit sums take: every int32 sum at its bound"""
    k = 32768
    a = np.full((3, k), 0x7e, np.uint8)
    b = np.full((k, 5), 0xfe, np.uint8)
    b[:, 1] = 0x01
    got = ops.quant_dot(dev(a), dev(b), fp8=True).cpu().numpy()
    assert np.array_equal(got, orc.quant_dot(a, b, orc.FP8).reshape(3, 5))


# the smallest M, N and K of the kernel, and slabs filled in part: short K reaches it in batches (alone it is
# left to the any-stride kernel)
@pytest.mark.parametrize("batch,m,n,k", [(1, 1, 5, 131), (1, 3, 4, 129), (500, 64, 67, 16), (500, 33, 35, 17),
                                         (500, 65, 66, 33), (300, 130, 65, 61)])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("fp8", [False, True])
def test_short_k_in_batches(ops, batch, m, n, k, trans_b, fp8):
    rng = np.random.default_rng(batch + n)
    assert kernel_of(m, n, k, trans_b=trans_b, fp8=fp8, batch=batch) == "ragged_exact"
    if fp8:
        a, b = _fp8(rng, (batch, m, k), False), _fp8(rng, (batch, k, n), False)
    else:
        a, b = (rng.integers(-128, 128, s, dtype=np.int8) for s in ((batch, m, k), (batch, k, n)))
    db = dev(np.ascontiguousarray(b.transpose(0, 2, 1))).transpose(1, 2) if trans_b else dev(b)
    print("short", batch, m, n, k, trans_b, fp8, flush=True)
    got = ops.quant_dot(dev(a), db, fp8=fp8).cpu().numpy()
    assert np.array_equal(got, orc.quant_dot(a, b, orc.FP8 if fp8 else orc.I8))
