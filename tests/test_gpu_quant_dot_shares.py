"""Split K in 128 x 128 tiles (a workspace, few tiles): edges of tiles, shares and slabs, against the product in
double; whole numbers exactly, fp8 by the bound of its float sums."""
import pytest
import torch

from tests.quant_dot_kernel import kernel_of, small_shares

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from amdmigraphx_amd import ops
    return ops


# one row and one 16-column tile; tiles begun in both directions; K an odd number of 64 (a prime one, 8128); shares of
# unequal length; the most tiles
@pytest.mark.parametrize("m,n,k,trans_b", [(1, 16, 4160, False), (1, 16, 8128, False), (20, 512, 4096, True), (130, 144, 4160, False), (127, 129, 4160, True),
                                           (257, 272, 4160, False), (33, 51, 4160, True), (40, 272, 8128, False), (128, 8192, 8256, False), (1000, 1008, 8256, False)])
@pytest.mark.parametrize("fp8", [False, True])
def test_against_the_product_in_double(ops, m, n, k, trans_b, fp8):
    need = ops.quant_dot_workspace_size(m, n, k, trans_b=trans_b, fp8=fp8)
    assert need > 0 and kernel_of(m, n, k, trans_b=trans_b, fp8=fp8, workspace=need) == "dma_shares"
    # (fp8 of 1 x 16 x 4160 goes to equal slices in 256 x 256 tiles)
    assert small_shares(m, n, k, trans_b=trans_b, fp8=fp8, workspace=need) > 1 or (fp8 and (m, n, k) == (1, 16, 4160))
    g = torch.Generator(device="cuda").manual_seed(m + n + k)

    def codes(*shape):
        if fp8:
            return (torch.randn(shape, generator=g, device="cuda") * 16).to(torch.float8_e4m3fn)
        return torch.randint(-128, 128, shape, generator=g, device="cuda", dtype=torch.int8)

    a, b = codes(m, k), (codes(n, k) if trans_b else codes(k, n))
    ad, bd = a.double(), (b.double().t() if trans_b else b.double())
    want = ad @ bd.contiguous()
    bits = (lambda t: t.view(torch.uint8)) if fp8 else (lambda t: t)
    right = bits(b).t() if trans_b else bits(b)
    room = torch.full((need + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    got = ops.quant_dot(bits(a), right, fp8=fp8, workspace=room[:need])
    assert bool((room[need:] == 0xA5).all())
    sa, sb = torch.rand(m, generator=g, device="cuda"), torch.rand(n, generator=g, device="cuda")
    scaled = ops.quant_dot(bits(a), right, fp8=fp8, workspace=room[:need], scale_a=sa, scale_b=sb)
    s = (sa[:, None] * sb).double()
    if not fp8:
        assert torch.equal(got.double(), want)
        assert torch.equal(scaled, (want * s).float())
        return
    # the instruction cuts products at a distance below the largest of a group: 2^-15 of the magnitudes' sum
    most = ad.abs() @ bd.abs().contiguous()
    assert bool(((got.double() - want).abs() <= torch.maximum(want.abs() * 1e-3, most * 2.0**-15)).all())
    assert bool(((scaled.double() - want * s).abs() <= torch.maximum((want * s).abs() * 1e-3, most * s * 2.0**-15)).all())


def test_nan_codes_stay_in_their_rows_and_columns(ops):
    """K an odd number of 64: what the last slab repeats of B brings no NaN into other columns"""
    m, n, k = 40, 144, 4160
    need = ops.quant_dot_workspace_size(m, n, k, fp8=True)
    assert need > 0
    a = torch.full((m, k), 0x38, dtype=torch.uint8, device="cuda")
    b = torch.full((k, n), 0x38, dtype=torch.uint8, device="cuda")
    a[7, 5], b[k - 1, 31], b[k - 100, 90] = 0x7F, 0xFF, 0x7F
    got = ops.quant_dot(a, b, fp8=True, workspace=torch.empty(need, dtype=torch.uint8, device="cuda"))
    nan = torch.zeros(m, n, dtype=torch.bool, device="cuda")
    nan[7, :], nan[:, 31], nan[:, 90] = True, True, True
    assert torch.equal(got.isnan(), nan) and bool((got[~nan] == k).all())
