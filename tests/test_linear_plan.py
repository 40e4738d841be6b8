"""Which kernel and tile the host picks (no GPU needed): the bf16-weight
layer."""
import ctypes

import pytest

from sllm_amd import _lib


def _bf16_plan(T, H, E, I, Is, k, aligned=1):
    if not _lib.available():
        pytest.fail(f"library not built: {_lib._lib_error}")
    out = (ctypes.c_int * 4)()
    assert _lib.lib().sllm_moe_bf16_plan_query(T, H, E, I, Is, k, aligned, out) == 0, _lib.last_error()
    return list(out)


@pytest.mark.parametrize("T", [1, 16, 64, 200, 1000])
@pytest.mark.parametrize("H,E,I,Is,k", [(1024, 16, 512, 512, 4), (2048, 32, 768, 0, 4)])
def test_unaligned_bf16_layer_keeps_the_gemvs_tiles(T, H, E, I, Is, k):
    """Weights below 16-byte alignment run on the GEMV, whose workgroups walk
    a tile's rows in fours: 16-row tiles, or 32 above 16 rows an expert (not
    the matrix-core kernel's 32 and 64)."""
    tile, bm, bound, _ = _bf16_plan(T, H, E, I, Is, k, aligned=0)
    assert (tile, bm) == (0, 32 if T * k > 16 * min(E, T * k) else 16)
    assert bound == _lib.lib().sllm_moe_tile_bound(T * k, E, bm)


def test_bf16_plan_rejects_bad_sizes():
    out = (ctypes.c_int * 4)()
    assert _lib.lib().sllm_moe_bf16_plan_query(4, 100, 8, 128, 0, 2, 1, out) == -1
    assert _lib.lib().sllm_moe_bf16_plan_query(4, 256, 8, 128, 0, 9, 1, out) == -1
