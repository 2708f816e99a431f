"""The workspace that mi355_w4a16_gemm_workspace_size names is one that the call can use (no GPU)."""
import os

import pytest

from amdmigraphx_amd import capi

pytestmark = pytest.mark.skipif(not os.path.exists(capi.lib_path()), reason="library not built in this checkout")


def _size(m, n, k):
    return capi.lib().mi355_w4a16_gemm_workspace_size(m, n, k, 128)


def test_no_room_for_weights_beyond_the_product_of_halves():
    """Offsets inside its operands are kept in 32 bits, so weights or activations of 2 GiB as halves are left to the
    tiles that dequantize for themselves: a size for them would be allocated and never used."""
    assert _size(2048, 131072 - 128, 8192) == 2 * (131072 - 128) * 8192
    assert _size(2048, 131072, 8192) == 0
    assert _size(2048, 128256, 16384) == 0
    assert _size(131072 - 128, 4096, 8192) == 2 * 4096 * 8192
    assert _size(131072, 4096, 8192) == 0


def test_room_for_many_rows_holds_two_bytes_a_weight():
    assert _size(2048, 14336, 4096) >= 2 * 14336 * 4096
    assert _size(2048, 14336, 1408) == 0  # shorter than the product's pipeline
