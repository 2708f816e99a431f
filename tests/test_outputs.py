"""What the functions of ops take as `out`, on the CPU: the library is replaced by a record of its calls, so that
what is refused is seen to be refused before anything could be stored."""
import pytest
import torch

from amdmigraphx_amd import ops


class _Record:
    """in the library's place: notes what is called and does nothing"""

    def __init__(self):
        self.called = []

    def __getattr__(self, name):
        def call(*args):
            self.called.append(name)
            return 0
        return call


@pytest.fixture
def library(monkeypatch):
    record = _Record()
    monkeypatch.setattr(ops, "lib", lambda: record)
    monkeypatch.setattr(ops, "_require_cuda", lambda *tensors: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    return record


def test_quant_dot_takes_wider_elements(library, monkeypatch):
    """results of 16 bits into a buffer of 32-bit elements: all of them fit, as they always did"""
    monkeypatch.setattr(torch.Tensor, "is_pinned", lambda self: True)  # as if the device could write it
    a, b, one = torch.ones(4, 64, dtype=torch.int8), torch.ones(64, 8, dtype=torch.int8), torch.ones(1)
    room = torch.empty(4, 8)
    assert ops.quant_dot(a, b, scale_a=one, out_dtype=torch.bfloat16, out=room) is room
    assert library.called == ["mi355_quant_dot"]


def _i8(*shape):
    return torch.ones(shape, dtype=torch.int8)


def _u8(*shape):
    return torch.ones(shape, dtype=torch.uint8)


def _call(name, out):
    """a result of 4 x 8 (with a batch of 3: 3 x 4 x 8)"""
    half = torch.ones(4, 256).half()
    return {"quant_dot": lambda: ops.quant_dot(_i8(4, 64), _i8(64, 8), out=out),
            "quant_dot batch": lambda: ops.quant_dot(_i8(3, 4, 64), _i8(3, 64, 8), out=out),
            "prepacked": lambda: ops.quant_dot_prepacked(_i8(4, 64), _u8(512), 8, out=out),
            "mx": lambda: ops.quant_dot_mx(_u8(4, 64), _u8(8, 64), torch.ones(4, 2), torch.ones(8, 2), out=out,
                                           workspace=_u8(16)),
            "mx batch": lambda: ops.quant_dot_mx(_u8(3, 4, 64), _u8(3, 8, 64), torch.ones(3, 4, 2), torch.ones(3, 8, 2), out=out,
                                                 workspace=_u8(16)),
            "w4": lambda: ops.w4a16_gemm(half, _u8(8, 128), torch.ones(8, 2).half(), 128, out=out),
            "w4 prepacked": lambda: ops.w4a16_gemm_prepacked(half, _u8(2048), 8, out=out)}[name]()


_TYPE = {"quant_dot": torch.int32, "prepacked": torch.int32, "mx": torch.float32, "w4": torch.float16}


@pytest.fixture
def pinned(monkeypatch):
    """host memory that the device may write"""
    monkeypatch.setattr(torch.Tensor, "is_pinned", lambda self: True)


@pytest.mark.parametrize("name", ["quant_dot", "quant_dot batch", "prepacked", "mx", "mx batch", "w4", "w4 prepacked"])
def test_an_output_holds_the_result(library, pinned, name):
    dtype = _TYPE[name.split()[0]]
    lead = (3,) if name.endswith("batch") else ()
    short, wide, more = lead + (3, 8), lead + (4, 24), lead + (9, 8)
    refused = [torch.empty(short, dtype=dtype), torch.empty(lead + (9, 24), dtype=dtype)[..., :3, :8]]
    if name != "prepacked":  # there the output's type is the result's, and the library says which it takes
        refused.append(torch.empty(lead + (4, 8), dtype=torch.int8))
    for out in refused:
        with pytest.raises(ops.Mi355Error, match="does not hold|narrower"):
            _call(name, out)
    if not lead:
        with pytest.raises(ops.Mi355Error):  # columns side by side in memory
            _call(name, torch.empty(8, 4, dtype=dtype).t())
    assert not any(c.startswith("mi355_") and not c.endswith("_size") for c in library.called)
    # what holds it: dense, rows of a wider tensor, more rows than the result has
    for out in (torch.empty(lead + (4, 8), dtype=dtype), torch.empty(wide, dtype=dtype)[..., 8:16], torch.empty(more, dtype=dtype)):
        library.called.clear()
        assert _call(name, out) is out
        assert library.called[-1].startswith("mi355_")


def test_an_output_lies_where_the_device_can_write(library):
    for name in ("quant_dot", "prepacked", "mx", "w4", "w4 prepacked"):
        with pytest.raises(ops.Mi355Error, match="device tensor"):
            _call(name, torch.empty(4, 8, dtype=_TYPE[name.split()[0]]))
    assert not any(not c.endswith("_size") for c in library.called)
