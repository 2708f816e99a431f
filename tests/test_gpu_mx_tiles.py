"""Block-scaled quant_dot with one float per block: the 64 x 64 tile kernel that reads the scales itself,
at the edges of its tiles and slabs, and the larger kernels where the rule hands over to them.
Operands whose sums are exact in float, so every kernel has to give the same bits."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from amdmigraphx_amd import ops
    return ops


def _operands(g, rows, k, fp4, batch):
    """codes, their values, and power-of-two block scales that keep every sum a whole multiple of 2^-5 below 2^19"""
    table = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], device="cuda", dtype=torch.float64)
    table = torch.cat([table, -table])
    if fp4:
        codes = torch.randint(0, 256, (batch, rows, k // 2), generator=g, device="cuda", dtype=torch.uint8)
        values = table[torch.stack([codes & 15, codes >> 4], dim=3).long()].reshape(batch, rows, k)
    else:
        v = torch.randint(-3, 4, (batch, rows, k), generator=g, device="cuda").float()
        codes, values = v.to(torch.float8_e4m3fn).view(torch.uint8), v.double()
    scales = torch.exp2(torch.randint(-1, 2, (batch, rows, k // 32), generator=g, device="cuda").float())
    return codes, values, scales


@pytest.mark.parametrize("batch,m,n,k", [(1, 1, 1, 128), (1, 64, 64, 256), (1, 65, 63, 384), (3, 130, 70, 640),
                                         (2, 17, 200, 1152), (1, 512, 4096, 512), (1, 1030, 2308, 4096)])
@pytest.mark.parametrize("fp4", [True, False])
def test_exact_sums(ops, batch, m, n, k, fp4):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, va, sa = _operands(g, m, k, fp4, batch)
    b, vb, sb = _operands(g, n, k, fp4, batch)
    print("mx", batch, m, n, k, fp4, flush=True)
    got = ops.quant_dot_mx(a, b, sa, sb, a_fp4=fp4, b_fp4=fp4)
    for i in range(batch):
        x = va[i] * sa[i].double().repeat_interleave(32, dim=1)
        w = vb[i] * sb[i].double().repeat_interleave(32, dim=1)
        assert torch.equal(got[i].double(), x @ w.t())


@pytest.mark.parametrize("fp4", [True, False])
@pytest.mark.parametrize("odd", [3.0, -1.0, 0.0, 2.0**-140, float("inf"), float("nan")])
def test_any_other_scale_takes_the_exact_path(ops, fp4, odd):
    """one scale of the last block of the last row that is no normal power of two"""
    m, n, k = 70, 66, 384
    g = torch.Generator(device="cuda").manual_seed(1)
    a, va, sa = _operands(g, m, k, fp4, 1)
    b, vb, sb = _operands(g, n, k, fp4, 1)
    sb[0, n - 1, k // 32 - 1] = odd
    got = ops.quant_dot_mx(a, b, sa, sb, a_fp4=fp4, b_fp4=fp4)[0].cpu().numpy()
    full = [s[0].repeat_interleave(32, dim=1).cpu().numpy() for s in (sa, sb)]
    x, w = ((v[0].float().cpu().numpy() * s).astype(np.float32) for v, s in zip((va, vb), full))
    want = orc.gemm(x, np.ascontiguousarray(w.T), orc.F32, orc.F32)
    assert np.array_equal(got, want.reshape(m, n), equal_nan=True)


@pytest.mark.parametrize("fp4", [True, False])
@pytest.mark.parametrize("m,n,k", [(40, 70, 512), (40, 70, 1024), (33, 97, 1152), (64, 64, 1408), (65, 40, 2176),
                                   (5, 65400, 256), (1990, 2047, 640)])
def test_scales_staged_for_four_slabs(ops, fp4, m, n, k):
    """one to four chunks of four slabs, whole and begun; the most tiles that stay with this kernel"""
    g = torch.Generator(device="cuda").manual_seed(m * n + k)
    a, va, sa = _operands(g, m, k, fp4, 1)
    b, vb, sb = _operands(g, n, k, fp4, 1)
    got = ops.quant_dot_mx(a, b, sa, sb, a_fp4=fp4, b_fp4=fp4)
    x = va[0] * sa[0].double().repeat_interleave(32, dim=1)
    w = vb[0] * sb[0].double().repeat_interleave(32, dim=1)
    assert torch.equal(got[0].double(), x @ w.t())


@pytest.mark.parametrize("fp4", [True, False])
def test_a_scale_of_any_quarter_and_chunk_raises_the_flag(ops, fp4):
    """A scale of 1.5 shows in one row or column only, and makes all sums exact: 2^-26 beside 2 is lost in float"""
    m, n, k = 64, 64, 1152 if fp4 else 640
    for is_b, row, block in ((0, 0, 0), (0, 31, 17), (0, 63, k // 32 - 1), (1, 1, 15), (1, 40, 16), (1, 63, 3)):
        g = torch.Generator(device="cuda").manual_seed(row + block)
        a, va, sa = _operands(g, m, k, fp4, 1)
        b, vb, sb = _operands(g, n, k, fp4, 1)
        (sb if is_b else sa)[0, row, block] = 1.5
        (sb if is_b else sa)[0, row - 1, block - 1] *= 2.0**-26
        got = ops.quant_dot_mx(a, b, sa, sb, a_fp4=fp4, b_fp4=fp4)
        x = (va[0] * sa[0].double().repeat_interleave(32, dim=1)).float().double()
        w = (vb[0] * sb[0].double().repeat_interleave(32, dim=1)).float().double()
        assert torch.equal(got[0], (x @ w.t()).float()), (is_b, row, block)


@pytest.mark.parametrize("batch,m,n,k", [(1, 40, 70, 512), (3, 33, 20, 256), (1, 2100, 4104, 4096)])
def test_rows_of_a_wider_output(ops, batch, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m)
    a, _, sa = _operands(g, m, k, False, batch)
    b, _, sb = _operands(g, n, k, False, batch)
    room = torch.full((batch, m + 1, n + 8), -1.0, device="cuda")
    out = room[:, :m, 4:4 + n]
    args = (a, b, sa, sb) if batch > 1 else (a[0], b[0], sa[0], sb[0])
    ops.quant_dot_mx(*args, out=out if batch > 1 else out[0])
    want = ops.quant_dot_mx(*args)
    assert torch.equal(out, want.view(batch, m, n))
    assert bool((room[:, m] == -1).all()) and bool((room[:, :, :4] == -1).all()) and bool((room[:, :, 4 + n:] == -1).all())
