"""Broadcast arithmetic whose columns run over several dimensions, and gathers of rows of every width, against torch."""
import ctypes

import pytest
import torch

from amdmigraphx_amd.capi import check, lib

pytestmark = pytest.mark.gpu


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("lens,a_dims,b_dims", [((3, 5, 8), "xxx", ".xx"), ((3, 5, 8), "xxx", "..x"), ((3, 5, 8), ".xx", "xxx"),
                                                ((3, 5, 8), "xx.", "xxx"), ((3, 5, 7), "xxx", ".xx"), ((2, 3, 4, 4), "xxxx", "x.xx"),
                                                ((2, 3, 4, 4), "xxxx", ".x.x"), ((2, 1, 6, 4), "xxxx", "x.xx"), ((1, 4, 1), "xxx", ".x."),
                                                ((2, 6, 2), "xx.", "xxx"), ((4, 6, 4), "...", "xxx"), ((7, 300, 12), "xxx", ".xx"),
                                                ((121, 226, 2, 4), "xxxx", "..xx"), ((50, 61, 4, 28), "xxxx", "..xx"), ((50, 61, 4, 32), "xxxx", "..xx"),
                                                ((30, 1, 5, 40), "xxxx", "x.x."), ((9, 11, 128), "xxx", "..x")])
def test_broadcast_add(lens, a_dims, b_dims):
    g = torch.Generator(device="cuda").manual_seed(sum(lens))

    def operand(dims):
        t = torch.randn([n if d == "x" else 1 for n, d in zip(lens, dims)], generator=g, device="cuda")
        return t, t.expand(lens)

    (ta, a), (tb, b) = operand(a_dims), operand(b_dims)
    strides = [[s if d == "x" else 0 for s, d in zip(t.stride(), dims)] for t, dims in ((ta, a_dims), (tb, b_dims))]
    arr = ctypes.c_int64 * len(lens)
    out = torch.full(lens, -1.0, device="cuda")
    for op, want in ((0, a + b), (1, a - b)):
        check(lib().mi355_binary_f32(op, _ptr(ta), arr(*strides[0]), _ptr(tb), arr(*strides[1]), _ptr(out), len(lens),
                                     arr(*lens), torch.cuda.current_stream().cuda_stream), "binary")
        assert torch.equal(out, want)


@pytest.mark.parametrize("words", [1, 3, 63, 64, 65, 252, 256, 260, 257, 768])
@pytest.mark.parametrize("kind", [torch.int32, torch.int64])
@pytest.mark.parametrize("shift", [0, 1])
def test_gather_rows(words, kind, shift):
    rows, n = 50, 37
    g = torch.Generator(device="cuda").manual_seed(words)
    room = torch.randn(rows * words + shift, generator=g, device="cuda")
    table = room[shift:].view(rows, words)
    ids = torch.randint(-rows, rows, (n,), generator=g, device="cuda").to(kind)
    ids[3], ids[5] = rows, -rows - 1  # outside: row 0
    out = torch.full((n + 1, words), -1.0, device="cuda")
    check(lib().mi355_gather_rows(_ptr(table), _ptr(ids), int(kind == torch.int64), _ptr(out), n, rows, words * 4,
                                  torch.cuda.current_stream().cuda_stream), "gather")
    at = torch.where((ids >= rows) | (ids < -rows), torch.zeros_like(ids), torch.where(ids < 0, ids + rows, ids)).long()
    assert torch.equal(out[:n], table[at]) and bool((out[n] == -1).all())


def _best(call):
    """shortest of 20 calls (ms)"""
    times = []
    for _ in range(20):
        start, stop = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        start.record()
        call()
        stop.record()
        stop.synchronize()
        times.append(start.elapsed_time(stop))
    return min(times)


def test_short_rows_are_no_workgroup_each():
    """a table of 2 x 4 added to a million of them: 2 times an ordinary sum's time, 8 times with a workgroup a row"""
    lens = (1118, 1118, 2, 4)
    x, t, out = torch.ones(lens, device="cuda"), torch.ones(2, 4, device="cuda"), torch.empty(lens, device="cuda")
    arr = ctypes.c_int64 * 4
    call = lambda: check(lib().mi355_binary_f32(0, _ptr(x), arr(*x.stride()), _ptr(t), arr(0, 0, 4, 1), _ptr(out), 4, arr(*lens),
                                                torch.cuda.current_stream().cuda_stream), "binary")
    assert _best(call) < 5 * _best(lambda: torch.add(x, x, out=out))


def _gather(table, ids, out):
    check(lib().mi355_gather_rows(_ptr(table), _ptr(ids), int(ids.dtype == torch.int64), _ptr(out), len(ids), len(table),
                                  table.shape[1] * 4, torch.cuda.current_stream().cuda_stream), "gather")


@pytest.mark.parametrize("n,words", [(1, 294912), (3, 100000), (3, 100001), (2, 1023), (5, 1024), (1, 1028), (70000, 64),
                                     (20000, 255), (20000, 1024 + 4)])
def test_gather_of_few_long_rows_and_many_short_ones(n, words):
    """a row in many pieces (whole and begun), and more pieces than there are waves"""
    rows = 40
    g = torch.Generator(device="cuda").manual_seed(words)
    table = torch.randn(rows, words, generator=g, device="cuda")
    ids = torch.randint(0, rows, (n,), generator=g, device="cuda")
    out = torch.full((n + 1, words), -1.0, device="cuda")
    _gather(table, ids, out)
    assert torch.equal(out[:n], table[ids]) and bool((out[n] == -1).all())


def test_one_long_row_is_copied_by_the_whole_chip():
    """A row of 5 MB takes about what a copy of it does; one wave by itself would take some hundred times that."""
    table, out = torch.ones(3, 1310720, device="cuda"), torch.empty(1, 1310720, device="cuda")
    ids = torch.tensor([1], device="cuda")

    assert _best(lambda: _gather(table, ids, out)) < 20 * _best(lambda: out.copy_(table[1:2]))
