"""quant_dot on both sides of the line between the kernels with 256 x 256 tiles and the register-staged
one: the shapes that stay with the large tiles, and those beside them that do not, against the same
product in float64 (exact for int8; the fp8 sums are float).  Each test says which kernel its calls run."""
import pytest
import torch

from tests.quant_dot_kernel import Forced, kernel_of

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from amdmigraphx_amd import ops
    return ops


def _codes(g, shape, fp8):
    if fp8:
        return (torch.randn(shape, generator=g, device="cuda") * 16).to(torch.float8_e4m3fn)
    return torch.randint(-128, 128, shape, generator=g, device="cuda", dtype=torch.int8)


def _check(ops, batch, m, n, k, trans_b, fp8, workspace=None, cut=2.0**-15):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = _codes(g, (batch, m, k), fp8)
    b = _codes(g, (batch, n, k) if trans_b else (batch, k, n), fp8)
    b = b.transpose(1, 2) if trans_b else b
    sa = torch.rand(1, generator=g, device="cuda") * 0.01
    sb = torch.rand(n, generator=g, device="cuda") * 0.01
    bits = (lambda t: t.view(torch.uint8)) if fp8 else (lambda t: t)
    bd = bits(b.transpose(1, 2)).transpose(1, 2) if trans_b else bits(b)
    print("route", batch, m, n, k, trans_b, fp8, flush=True)
    got = [ops.quant_dot(bits(a), bd, fp8=fp8), ops.quant_dot(bits(a), bd, fp8=fp8, scale_a=sa, scale_b=sb)]
    if batch == 1:
        need = ops.quant_dot_workspace_size(m, n, k, trans_b=trans_b, fp8=fp8)
        if need:
            got.append(ops.quant_dot(bits(a)[0], bd[0], fp8=fp8, scale_a=sa, scale_b=sb,
                                     workspace=torch.empty(need, dtype=torch.uint8, device="cuda"))[None])
    for i in range(batch):
        acc = a[i].double() @ b[i].double().contiguous()
        s = (sa * sb).double()
        for t, want in zip(got, [acc, acc * s, acc * s]):
            if not fp8:
                assert torch.equal(t[i].double(), want.float().double() if t.is_floating_point() else want)
                continue
            # the contract of the fp8 sums: 1e-3 relative, or, where a sum cancels, 2^-15 of the sum of the
            # magnitudes (the instruction cuts its products at a distance below the largest of them; both
            # kernels are 1.46e-5 from the exact sums as a whole)
            most = (a[i].double().abs() @ b[i].double().abs().contiguous()) * (s if want is not acc else 1.0)
            assert bool(((t[i].double() - want).abs() <= torch.maximum(want.abs() * 1e-3, most * cut)).all())


def _kernels(batch, m, n, k, trans_b, fp8):
    """of the bare product, with scales, and with a workspace as well"""
    room = dict(out="f32", workspace=1 << 30) if batch == 1 else dict(out="f32")
    return {kernel_of(m, n, k, trans_b=trans_b, fp8=fp8, batch=batch, **kw) for kw in (dict(), dict(out="f32"), room)}


# K on both sides of the four-wave kernels' first length; edges of the 256 tiles
@pytest.mark.parametrize("batch,m,n,k", [(1, 4100, 4112, 1600), (1, 2050, 8208, 3136), (2, 4100, 2064, 3136)])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("fp8", [False, True])
def test_large_tiles(ops, batch, m, n, k, trans_b, fp8):
    assert _kernels(batch, m, n, k, trans_b, fp8) == {"dma"}
    _check(ops, batch, m, n, k, trans_b, fp8)


# K that is no multiple of 64
@pytest.mark.parametrize("batch,m,n,k", [(1, 4100, 8240, 2064), (2, 4100, 4112, 2096)])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("fp8", [False, True])
def test_large_register_staged_tiles(ops, batch, m, n, k, trans_b, fp8):
    assert _kernels(batch, m, n, k, trans_b, fp8) == {"mfma"}
    _check(ops, batch, m, n, k, trans_b, fp8)


# few tiles of a long K: in shares where there is room or the product is bare, register-staged without
@pytest.mark.parametrize("batch,m,n,k", [(1, 16, 512, 8192), (1, 16, 16, 3072), (1, 37, 272, 25600)])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("fp8", [False, True])
def test_long_k_of_few_tiles(ops, batch, m, n, k, trans_b, fp8):
    assert _kernels(batch, m, n, k, trans_b, fp8) == {"ragged" if fp8 else "dma_atomic", "ragged", "dma_shares"}
    _check(ops, batch, m, n, k, trans_b, fp8)


# tiles of 64 x 64, and of 128 x 128 where those fill the chip (2060 x 2064)
@pytest.mark.parametrize("batch,m,n,k", [(5, 64, 64, 64), (3, 197, 208, 128), (2, 130, 80, 272), (40, 384, 64, 384),
                                         (1, 2060, 2064, 784), (1, 1030, 1040, 1024), (1, 300, 2064, 1088)])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("fp8", [False, True])
def test_small_tiles(ops, batch, m, n, k, trans_b, fp8):
    assert _kernels(batch, m, n, k, trans_b, fp8) == {"ragged"}
    _check(ops, batch, m, n, k, trans_b, fp8)


# all of K in one slab: K at and around 16, 64 and 128, rows and columns that end inside a tile, more tiles than
# a CU holds at once
@pytest.mark.parametrize("batch,m,n,k", [(1, 1, 4, 16), (3, 65, 63, 17), (2, 64, 64, 64), (2, 130, 70, 65), (1, 197, 197, 100),
                                         (40, 33, 191, 128), (96, 197, 197, 64), (2, 70, 66, 129)])
@pytest.mark.parametrize("fp8", [False, True])
def test_one_slab(ops, batch, m, n, k, fp8):
    # (3 x 65 x 63 x 17 and the like are there for what lies beside the kernel: see below for the calls that reach it)
    _check(ops, batch, m, n, k, True, fp8, cut=_cut(batch, m, n, k, fp8))


def _cut(batch, m, n, k, fp8):
    """One instruction cuts each of up to 128 products 20 bits below the largest of them, which is at most the sum of
    the magnitudes: 2^-13 of that.  (Among the millions of sums of 96 x 197 x 197 some reach 2^-14, the same bits as
    the 256 x 256 kernels'.)  The other kernels' sums keep the narrower bound, those in digits are exact."""
    return 2.0**-13 if fp8 and "ragged" in _kernels(batch, m, n, k, True, fp8) else 2.0**-15


# the kernel itself: int8 whatever K is, e4m3fn in float where rows are whole 16-byte pieces and N whole groups of 4
@pytest.mark.parametrize("batch,m,n,k", [(20, 129, 132, 16), (9, 131, 192, 48), (5, 300, 500, 64), (9, 131, 188, 80),
                                         (12, 197, 196, 112), (3, 70, 64, 128)])
@pytest.mark.parametrize("fp8", [False, True])
def test_one_slab_of_whole_pieces(ops, batch, m, n, k, fp8):
    assert _kernels(batch, m, n, k, True, fp8) == {"ragged"}
    _check(ops, batch, m, n, k, True, fp8, cut=_cut(batch, m, n, k, fp8))


@pytest.mark.parametrize("batch,m,n,k", [(5, 300, 500, 17), (5, 300, 501, 33), (9, 131, 190, 63), (5, 300, 499, 65),
                                         (12, 197, 197, 111), (2, 130, 70, 127)])
def test_one_slab_of_any_bytes(ops, batch, m, n, k):
    assert _kernels(batch, m, n, k, True, False) == {"ragged_exact"}
    _check(ops, batch, m, n, k, True, False)


# results within one and a half of the last-level cache and beyond (one slab and not; whole lines; mostly padding
# otherwise; several matrices), rows that are no whole groups of 4
@pytest.mark.parametrize("batch,m,n,k", [(1, 4200, 4304, 80), (1, 9400, 9500, 48), (1, 9400, 9504, 64), (300, 64, 1000, 64),
                                         (5, 4300, 4204, 128), (3, 882, 881, 64), (1, 700, 1503, 128)])
@pytest.mark.parametrize("fp8", [False, True])
def test_short_k_of_many_tiles(ops, batch, m, n, k, fp8):
    _check(ops, batch, m, n, k, True, fp8, cut=_cut(batch, m, n, k, fp8))


@pytest.mark.parametrize("batch,m,n,k", [(96, 197, 197, 64), (3, 300, 260, 128), (1, 500, 1030, 128)])
@pytest.mark.parametrize("out", [None, torch.float32, torch.bfloat16])
def test_one_slab_gives_the_bits_of_the_large_tiles(ops, monkeypatch, batch, m, n, k, out):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, b = (_codes(g, (batch, rows, k), True).view(torch.uint8) for rows in (m, n))
    kw = dict(fp8=True, out_dtype=out, **(dict(scale_a=torch.rand(1, generator=g, device="cuda")) if out else {}))
    assert kernel_of(m, n, k, trans_b=True, fp8=True, batch=batch, out="f32" if out else None) == "ragged"
    got = ops.quant_dot(a, b.transpose(1, 2), **kw)
    large = Forced("dma")
    monkeypatch.setattr(ops, "lib", lambda: large)
    want = ops.quant_dot(a, b.transpose(1, 2), **kw)
    assert large.taken == 1 and torch.equal(got, want)
