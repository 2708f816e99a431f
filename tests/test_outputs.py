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


def test_quant_dot_takes_wider_elements(library):
    """results of 16 bits into a buffer of 32-bit elements: all of them fit, as they always did"""
    a, b, one = torch.ones(4, 64, dtype=torch.int8), torch.ones(64, 8, dtype=torch.int8), torch.ones(1)
    room = torch.empty(4, 8)
    assert ops.quant_dot(a, b, scale_a=one, out_dtype=torch.bfloat16, out=room) is room
    assert library.called == ["mi355_quant_dot"]
