"""int4 weight-only GEMM of many rows: weights dequantized into the workspace, then the 256 x 256
half kernel.  Against a float64 product of the dequantized half weights."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from amdmigraphx_amd import ops
    return ops


# rows and columns that fill no 256 x 256 tile, K of 12 * 4 slabs, one more trip of slabs and a remainder; N no
# multiple of 128: 16, 144 and 240 columns of the last tile, one part of K and four
@pytest.mark.parametrize("m,n,k,pad", [(1999, 7296, 1536, 0), (970, 15744, 1664, 8), (2048, 8192, 2688, 0),
                                       (1000, 3968, 9216, 8), (1999, 7184, 1536, 8), (970, 15760, 1664, 0),
                                       (512, 4112, 8192, 8), (700, 4080, 8192, 0)])
@pytest.mark.parametrize("group,zeros", [(128, "scalar"), (64, "group"), (32, "packed")])
def test_many_rows(ops, m, n, k, pad, group, zeros):
    need = ops.w4a16_gemm_workspace_size(m, n, k, group)
    assert need >= 2 * n * k  # the shapes of this test take the two passes
    assert (need > 2 * n * k) == (k > 4096)  # the last one with K in shares
    rng = np.random.default_rng(m + group)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float16)).cuda()
    packed = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
    scales = orc.half_from_f32(rng.uniform(0.005, 0.02, (n, k // group)).astype(np.float32))
    scales[::17, 0] = 0x0001  # a subnormal scale
    groups = k // group
    z = rng.integers(0, 16, (n, groups), dtype=np.uint8)
    if zeros == "scalar":
        z[:] = 8
        zp, mode = 8, None
    elif zeros == "group":
        zp, mode = torch.from_numpy(z).cuda(), ops.W4ZP.GROUP
    else:
        both = np.concatenate([z, np.zeros((n, groups % 2), np.uint8)], axis=1)
        zp, mode = torch.from_numpy(both[:, ::2] | (both[:, 1::2] << 4)).cuda().contiguous(), ops.W4ZP.PACKED
    q = np.stack([packed & 15, packed >> 4], axis=2).reshape(n, groups, group).astype(np.float32)
    w = (q - z[:, :, None].astype(np.float32)) * orc.half_to_f32(scales)[:, :, None]
    w = torch.from_numpy(orc.half_from_f32(w.reshape(n, k)).view(np.float16)).cuda().double()
    out = torch.full((m, n + pad), -1.0, dtype=torch.float16, device="cuda")
    got = ops.w4a16_gemm(x, torch.from_numpy(packed).cuda(), torch.from_numpy(scales.view(np.float16)).cuda(), group,
                         zp, zp_mode=mode, out=out[:, :n], workspace=torch.empty(need, dtype=torch.uint8, device="cuda"))
    want = x.double() @ w.t()
    # k float32 additions round to nearest, the result is cut to 11 bits (subnormal steps of 2^-24 below)
    bound = (x.double().abs() @ w.t().abs()) * (k * 2.0**-24) + want.abs() * 2.0**-10 + 2.0**-24
    assert bool(((got.double() - want).abs() <= bound).all())
    assert pad == 0 or bool((out[:, n:] == -1).all())


def test_a_workspace_one_byte_short_is_left_alone(ops):
    """the call falls back to the tiles that dequantize for themselves, with the same result up to the order of sums"""
    m, n, k, group = 1000, 3968, 9216, 128
    need = ops.w4a16_gemm_workspace_size(m, n, k, group)
    assert need > 2 * n * k
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(m, k, generator=g, device="cuda").half()
    w = torch.randint(0, 256, (n, k // 2), generator=g, dtype=torch.uint8, device="cuda")
    scales = (torch.rand(n, k // group, generator=g, device="cuda") * 0.015 + 0.005).half()
    room = torch.full((need,), 0x5a, dtype=torch.uint8, device="cuda")
    short = ops.w4a16_gemm(x, w, scales, group, workspace=room[:-1])
    assert bool((room == 0x5a).all())
    whole = ops.w4a16_gemm(x, w, scales, group, workspace=room)
    assert not bool((room[:2 * n * k] == 0x5a).all())
    # k float32 additions in either order, and the cut to 11 bits twice
    dense = torch.stack([w & 15, w >> 4], dim=2).reshape(n, -1, group).float() - 8
    dense = (dense * scales.float()[:, :, None]).reshape(n, k).abs().double()
    bound = 2 * (x.double().abs() @ dense.t()) * (k * 2.0**-24) + whole.double().abs() * 2.0**-9 + 2.0**-23
    assert bool(((short.double() - whole.double()).abs() <= bound).all())


def test_infinities_nan_and_results_beyond_half(ops):
    """In activations and scales, and sums outside the half range: as the definition has them, and as the call
    without a workspace, whose kernel dequantizes for itself."""
    m, n, k, group = 970, 15744, 1664, 128
    need = ops.w4a16_gemm_workspace_size(m, n, k, group)
    assert need == 2 * n * k
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(m, k, generator=g, device="cuda").half()
    w = torch.randint(0, 256, (n, k // 2), generator=g, dtype=torch.uint8, device="cuda")
    w[:, 0] = 0x88  # the first two weights are zero
    w[1, 5] = 0x8f
    scales = (torch.rand(n, k // group, generator=g, device="cuda") * 0.015 + 0.005).half()
    x[3, 10], x[5, k - 1], x[7, 0], x[8, 11] = float("inf"), float("-inf"), float("inf"), float("nan")
    x[20:40] *= 3000
    scales[100, 2], scales[101, 0], scales[102, 3], scales[200, 1] = float("inf"), float("inf"), float("nan"), 65504.0
    scales[300:310] *= 4000
    dense = torch.stack([w & 15, w >> 4], dim=2).reshape(n, -1, group).double() - 8
    dense = (dense * scales.double()[:, :, None]).reshape(n, k)
    # a weight beyond half's range is cut to its largest value
    dense = torch.where(dense.isfinite(), dense.clamp(-65504, 65504), dense)
    # rounded toward zero, as dequantizelinear rounds it
    near = dense.half()
    away = near.double().abs() > dense.abs()
    near = torch.where(away, (near.view(torch.int16) - 1).view(torch.float16), near)
    want = x.double() @ near.double().t()
    got = ops.w4a16_gemm(x, w, scales, group, workspace=torch.empty(need, dtype=torch.uint8, device="cuda")).double()
    tiles = ops.w4a16_gemm(x, w, scales, group).double()
    for result in (got, tiles):
        assert bool((result.isnan() == want.isnan()).all())
        assert bool((result == want)[want.isinf()].all())
    assert bool(want.isnan().any()) and bool(want.isinf().any())
    fin = want.isfinite()
    # of the sums that leave the range for certain both make the same
    over = fin & (want.abs() > 66000)
    assert bool(over.any()) and bool((got == tiles)[over].all())
    size = torch.where(x.isfinite(), x, torch.zeros_like(x)).double().abs() @ \
        torch.where(near.isfinite(), near, torch.zeros_like(near)).double().abs().t()
    bound = size * (k * 2.0**-24) + want.abs() * 2.0**-10 + 2.0**-24
    within = fin & (want.abs() + bound < 65504)
    for result in (got, tiles):
        assert bool(((result - want).abs() <= bound)[within].all())
