"""Scales, zero points, column and row sums that are views with a stride give what their dense copies give."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from amdmigraphx_amd import ops
    return ops


def _strided(t):
    """the same values, every third element of a larger tensor (of every row, for a matrix)"""
    wide = torch.zeros(t.shape + (3,), dtype=t.dtype, device=t.device)
    wide[..., 1] = t
    view = wide[..., 1]
    assert torch.equal(view, t) and (t.numel() == 1 or not view.is_contiguous())
    return view


def _codes(g, *shape):
    return torch.randint(-128, 128, shape, generator=g, device="cuda", dtype=torch.int8)


@pytest.mark.parametrize("m,n,k", [(100, 96, 128), (70, 30, 65)])
def test_quant_dot(ops, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(1)
    a, b = _codes(g, m, k), _codes(g, k, n)
    sa, sb = (torch.rand(s, generator=g, device="cuda") * 0.01 + 0.001 for s in (m, n))
    sums = dict(colsum_b=ops.colsum_i8(b), rowsum_a=ops.rowsum_i8(a))
    want = ops.quant_dot(a, b, scale_a=sa, scale_b=sb, zp_a=3, zp_b=-5, **sums)
    got = ops.quant_dot(a, b, scale_a=_strided(sa), scale_b=_strided(sb), zp_a=3, zp_b=-5,
                        **{name: _strided(t) for name, t in sums.items()})
    assert torch.equal(got, want)


def test_quant_dot_prepacked(ops):
    g = torch.Generator(device="cuda").manual_seed(2)
    m, n, k = 5, 512, 1024
    a, b = _codes(g, m, k), _codes(g, k, n)
    packed = ops.quant_dot_prepack(b)
    sa, sb = (torch.rand(s, generator=g, device="cuda") * 0.01 + 0.001 for s in (m, n))
    bias, colsum = torch.randn(n, generator=g, device="cuda"), ops.colsum_i8(b)
    want = ops.quant_dot_prepacked(a, packed, n, scale_a=sa, scale_b=sb, zp_a=3, colsum_b=colsum, bias=bias)
    got = ops.quant_dot_prepacked(a, packed, n, scale_a=_strided(sa), scale_b=_strided(sb), zp_a=3,
                                  colsum_b=_strided(colsum), bias=_strided(bias))
    assert torch.equal(got, want)


def test_quant_convolution(ops):
    g = torch.Generator(device="cuda").manual_seed(3)
    x, w = _codes(g, 2, 16, 9, 9), _codes(g, 32, 16, 3, 3)
    sx, sw = torch.full((1,), 0.02, device="cuda"), torch.rand(32, generator=g, device="cuda") * 0.01 + 0.001
    want = ops.quant_convolution(x, w, padding=(1, 1), scale_x=sx, scale_w=sw)
    assert torch.equal(ops.quant_convolution(x, w, padding=(1, 1), scale_x=sx, scale_w=_strided(sw)), want)


@pytest.mark.parametrize("m", [1, 40])
def test_w4a16(ops, m):
    g = torch.Generator(device="cuda").manual_seed(4)
    n, k, group = 256, 512, 128
    x = torch.randn(m, k, generator=g, device="cuda").half()
    w = torch.randint(0, 256, (n, k // 2), generator=g, device="cuda", dtype=torch.uint8)
    scales = (torch.rand(n, k // group, generator=g, device="cuda") * 0.01).half()
    zp = torch.randint(0, 16, (n, k // group), generator=g, device="cuda", dtype=torch.uint8)
    want = ops.w4a16_gemm(x, w, scales, group, zp)
    assert torch.equal(ops.w4a16_gemm(x, _strided(w), _strided(scales), group, _strided(zp)), want)
