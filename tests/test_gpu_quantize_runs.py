"""the kernels that quantize, dequantize (16, 4 or 2 elements a thread), pack and unpack (8 bytes), at the
lengths and addresses where runs overlap or are misaligned, against the CPU oracle: all bit for bit."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

_FLOATS = {"f32": (orc.F32, torch.float32, np.uint32), "f16": (orc.F16, torch.float16, np.uint16),
           "bf16": (orc.BF16, torch.bfloat16, np.uint16)}
_CODES = {"int8": (orc.I8, np.int8), "uint8": (orc.U8, np.uint8), "fp8": (orc.FP8, np.uint8)}


@pytest.fixture(scope="module")
def ops():
    from amdmigraphx_amd import ops
    return ops


def _bits(x, kind):
    """float32 values as numpy carries them for the oracle: themselves, or the bits of the 16-bit type"""
    return {"f32": lambda v: v, "f16": orc.half_from_f32, "bf16": orc.bf16_from_f32}[kind](np.float32(x))


def _put(bits, dtype=None, shift=0):
    """the bits on the device, `shift` elements behind an aligned address"""
    flat = torch.zeros(bits.size + shift, dtype=torch.from_numpy(bits.reshape(-1)[:0]).dtype)
    flat[shift:] = torch.from_numpy(np.ascontiguousarray(bits).reshape(-1))
    flat = flat.cuda() if dtype is None else flat.cuda().view(dtype)
    return flat[shift:].view(bits.shape)


def _put_float(bits, kind, shift=0):
    _, dtype, raw = _FLOATS[kind]
    signed = {np.uint32: np.int32, np.uint16: np.int16}[raw]
    return _put(np.ascontiguousarray(bits).view(signed), dtype, shift)


def _param(rng, place, rows, cols, make):
    n = {"tensor": 1, "row": rows, "col": cols, "full": rows * cols}[place]
    v = make(n)
    return v.reshape(rows, cols) if place == "full" else v


@pytest.mark.parametrize("rows,cols,shift", [(1, 1, 0), (3, 7, 1), (5, 8, 0), (2, 9, 3), (37, 101, 1), (300, 15, 5),
                                             (5, 16, 2), (2, 33, 0), (17, 4096, 0), (1, 70001, 1), (50, 1, 1), (40, 2, 0), (33, 3, 1),
                                             (20, 4, 2), (21, 5, 0), (9, 17, 1), (700, 31, 0)])
@pytest.mark.parametrize("place", ["tensor", "row", "col", "full"])
@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
def test_runs_there_and_back(ops, kind, place, rows, cols, shift):
    _there_and_back(ops, kind, place, rows, cols, shift)


# 2^21 elements and more with one parameter for a row: 16 elements a thread
@pytest.mark.parametrize("place,rows,cols,shift", [("tensor", 1, 2097157, 3), ("tensor", 3, 699053, 0), ("row", 131, 16111, 1),
                                                   ("row", 116509, 18, 0), ("row", 131073, 16, 1)])
@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
def test_long_runs_there_and_back(ops, kind, place, rows, cols, shift):
    _there_and_back(ops, kind, place, rows, cols, shift)


def _there_and_back(ops, kind, place, rows, cols, shift):
    rng = np.random.default_rng(rows * cols + shift)
    x = rng.standard_normal((rows, cols)) * rng.choice([0.01, 1.0, 30.0], (rows, cols))
    odd = np.array([0.0, -0.0, 0.5, -2.5, 1e9, -1e9, np.inf, -np.inf, np.nan, 1e-30, -1e-30])
    at = rng.integers(0, x.size, min(len(odd), x.size))
    x.reshape(-1)[at] = odd[:len(at)]
    x = _bits(x, kind)
    ft = _FLOATS[kind][0]
    scale = _bits(_param(rng, place, rows, cols, lambda n: rng.uniform(0.01, 0.5, n)), kind)
    dx, ds = _put_float(x, kind, shift), _put_float(scale, kind, shift)
    for code, (ct, np_code) in _CODES.items():
        lo, hi = {"int8": (-128, 128), "uint8": (0, 256), "fp8": (0, 0x60)}[code]
        zp = _param(rng, place, rows, cols, lambda n: rng.integers(lo, hi, n)).astype(np_code)
        for z in (None, zp):
            dz = None if z is None else _put(z, shift=shift)
            # fp8 with a zero point is quantized by the kernel of any strides
            want = orc.quantizelinear(x, scale, z, ft, ct)
            got = ops.quantizelinear(dx, ds, dz, ct)
            assert np.array_equal(got.cpu().numpy().view(np_code), want), (code, z is None)
            codes = rng.integers(0, 256, (rows, cols)).astype(np.uint8).view(np_code)
            if code == "fp8":
                codes &= 0xf7  # no NaN: its payload is not part of the contract
            want = orc.dequantizelinear(codes, scale, z, ct, ft)
            got = ops.dequantizelinear(_put(codes, shift=shift), ds, dz, ct)
            raw = _FLOATS[kind][2]
            back = got.cpu().contiguous().view(torch.int32 if raw == np.uint32 else torch.int16).numpy().view(raw)
            assert np.array_equal(back, np.ascontiguousarray(want).view(raw)), (code, z is None)


@pytest.mark.parametrize("count,shift", [(1, 0), (7, 1), (8, 0), (9, 3), (15, 1), (2047, 0), (4099, 1)])
@pytest.mark.parametrize("dtype", [np.uint8, np.int8])
def test_int4_runs(ops, dtype, count, shift):
    rng = np.random.default_rng(count)
    codes = rng.integers(0, 256, (1, 2 * count)).astype(np.uint8).view(dtype)
    assert np.array_equal(ops.pack_int4(_put(codes, shift=shift)).cpu().numpy(), orc.pack_int4(codes))
    packed = rng.integers(0, 256, (1, count)).astype(np.uint8).view(dtype)
    assert np.array_equal(ops.unpack_int4(_put(packed, shift=shift)).cpu().numpy(), orc.unpack_int4(packed))


def test_fp8_zeros_and_extremes_keep_their_signs(ops):
    """-0 / s becomes +0 in the operator's double sum, a negative quotient below the range stays -0"""
    x = np.float32([[0.0, -0.0, -1e-30, 1e-30, -1e-38, np.inf, -np.inf, np.nan, -3.0, 3.0, -5.0, 447.0]])
    for s in (1.0, 1e20, np.inf, 1e-30, 0.0):
        want = orc.quantizelinear(x, np.float32(s), None, orc.F32, orc.FP8)
        got = ops.quantizelinear(_put(x), torch.tensor([s], device="cuda"), None, ops.DT.FP8)
        assert np.array_equal(got.cpu().numpy(), want), s


def _near_ties(rng, scale, kind):
    """values around scale * (whole + 1/2), where the last bit of the quotient decides, and at the bounds of the range
    in which the quotient is made from the reciprocal"""
    whole = np.arange(-130, 260)
    with np.errstate(over="ignore", invalid="ignore"):
        t = (np.float64(scale) * (whole + 0.5)).astype(np.float32)
        x = [np.nextafter(t, np.float32(-np.inf)), t, np.nextafter(t, np.float32(np.inf))]
        x.append((np.float64(scale) * rng.uniform(-500, 500, 300)).astype(np.float32))
        x.append((np.float64(scale) * 2.0**rng.uniform(-40, 10, 300)).astype(np.float32))
        x.append(np.float32([2.0**60, np.nextafter(np.float32(2**60), np.float32(0)), -2.0**60, 2.0**-149, -2.0**-126, 0, -0.0]))
        x = np.concatenate(x)
    return _bits(np.where(np.isfinite(x), x, np.float32(1)), kind)


@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
def test_quotients_by_the_reciprocal(ops, kind):
    """One scale for a tensor: the quotient is the corrected product with the reciprocal for scales of 2^-60 to 2^60 and
    values up to 2^60, else a division, and has to be the division's in every case."""
    rng = np.random.default_rng(11)
    lo, hi = np.float32(2.0**-60), np.float32(2.0**60)
    scales = [lo, np.nextafter(lo, np.float32(0)), np.nextafter(lo, hi), hi, np.nextafter(hi, lo),
              np.nextafter(hi, np.float32(np.inf)), 2.0**-140, 2.0**100, 1.0, np.nextafter(np.float32(1), lo),
              np.nextafter(np.float32(2), lo), -0.37]
    scales += [m * 2.0**e for m, e in zip(rng.uniform(1, 2, 60), rng.integers(-14, 15, 60))]
    if kind == "f32":
        scales += [m * 2.0**e for m, e in zip(rng.uniform(1, 2, 60), rng.integers(-62, 62, 60))]
    for s in scales:
        sb = _bits(np.float32([s]), kind)
        if kind == "f16" and not 6e-8 <= abs(float(orc.half_to_f32(sb)[0])) <= 65504:
            continue
        x = _near_ties(rng, np.float32(s), kind).reshape(1, -1)
        # once in runs of 4, and once in runs of 16 (2^21 elements and more)
        for repeat in (1, (1 << 21) // x.size + 1) if s in (lo, hi, 1.0, -0.37) else (1,):
            y = np.ascontiguousarray(np.tile(x, (1, repeat)))
            dx, ds = _put_float(y, kind), _put_float(sb, kind)
            for code, (ct, np_code) in _CODES.items():
                want = orc.quantizelinear(x, sb, None, _FLOATS[kind][0], ct)
                got = ops.quantizelinear(dx, ds, None, ct).cpu().numpy().view(np_code)
                assert np.array_equal(got, np.tile(want, (1, repeat))), (float(s), code, repeat)
