"""quant_dot's choice of a kernel, asked on the host (no GPU)."""
import os

import pytest

from amdmigraphx_amd import capi
from tests.quant_dot_kernel import kernel_of

pytestmark = pytest.mark.skipif(not os.path.exists(capi.lib_path()), reason="library not built in this checkout")


def test_register_staged_kernel_keeps_room_for_its_read_ahead():
    """It counts K in ints and asks for positions up to two slabs of 256 and 240 bytes behind the last slab: with
    K up to 767 short of 2^31 such a position would wrap around to an address far in front of the matrix."""
    for k in (2**31 - 256, 2**31 - 257, 2**31 - 767, 2**31 - 1023, 2**31 - 1024):
        assert kernel_of(1, 1, k, trans_b=True) == "generic"
    last = 2**31 - 1025
    furthest = ((last + 255) // 256 + 1) * 256 + 240
    assert furthest < 2**31
    assert kernel_of(1, 1, last, trans_b=True) == "ragged_exact"


def test_register_staged_kernel_keeps_to_the_largest_grid():
    """2^24 workgroups of 256 threads are more than one launch takes; 180 GB of bfloat16 results still fit the card."""
    m = 300001
    assert (m + 63) // 64 * ((m + 63) // 64) * 256 >= 2**32
    assert kernel_of(m, m, 17, fp8=True, out="bf16") == "generic"
    assert kernel_of(250001, 250001, 17, fp8=True, out="bf16") == "ragged_exact"
    assert (m + 127) // 128 * ((m + 127) // 128) * 256 < 2**32
    assert kernel_of(m, m, 17, out="bf16") == "ragged_exact"
