"""Which kernel and tile the host picks (no GPU needed): the bf16-weight
layer, the FP8 and MXFP4 linears (at 256 CUs)."""
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


# tokens below / from the line in rows a touched expert
@pytest.mark.parametrize("H,E,I,Is,k,below,above", [
    (2048, 32, 768, 0, 4, (1, 3, 8, 24), (32, 64)), (2048, 128, 768, 0, 8, (1, 32, 48), (64,)),
    (2048, 1, 5632, 0, 1, (1, 2), (3, 4)), (4096, 8, 14336, 0, 2, (1, 12), (16,)),
    # a shared expert, whose launches of its own cost more beside few weights
    (2048, 512, 512, 512, 10, (2, 3, 64), (1, 130)), (1024, 16, 512, 512, 4, (), (1, 8, 64)),
    (2048, 32, 768, 768, 4, (2, 6, 12), (1, 5, 16, 24))])
def test_bf16_layer_kernel_by_rows(H, E, I, Is, k, below, above):
    """Few rows a touched expert run on the GEMV: below 3.4 (one expert 3,
    beside a shared one 2.25 and enough weights)."""
    for T in below:
        tile, bm, bound, sh = _bf16_plan(T, H, E, I, Is, k)
        assert tile == 0 and bm == (32 if T * k > 16 * min(E, T * k) else 16), T
        assert bound == _lib.lib().sllm_moe_tile_bound(T * k, E, bm)
        assert (sh > 0) == (Is > 0 and T >= 3), T
    for T in above:
        tile, bm, _, sh = _bf16_plan(T, H, E, I, Is, k)
        assert tile > 0 and bm == {1: 16, 2: 32, 3: 32, 4: 64}[tile] and sh == 0, T


def _workspace(T, H, E, I, Is, k, logits_given):
    a = _lib.QwenArgs()
    a.T, a.H, a.E, a.I, a.Is, a.topk, a.wdtype = T, H, E, I, Is, k, 1
    a.su = 8 if Is else None
    a.logits_given = logits_given
    return _lib.lib().sllm_moe_qwen_workspace_bytes(ctypes.byref(a))


@pytest.mark.parametrize("T", [65, 130, 1000, 4000])
@pytest.mark.parametrize("logits_given", [0, 1])
@pytest.mark.parametrize("H,E,I,Is,k", [(1024, 16, 512, 512, 4), (2048, 32, 768, 0, 4),
                                        (7168, 256, 2048, 2048, 8), (2048, 512, 512, 512, 10)])
def test_bf16_workspace_holds_no_router_slices(T, H, E, I, Is, k, logits_given):
    """Above 64 tokens the workspace is that of the unsplit router (a call at
    the limit of the fixed scratch stays within it): routing tables, h, y."""
    N, al = T * k, lambda b: -(-b // 256) * 256
    bm = 32 if N > 16 * min(E, N) else 16
    tables = [T * E * 4 * (1 - logits_given), N * 4, N * 4, E * 4, (E + 1) * 4, N * 4, N * 4,
              N * 4, _lib.lib().sllm_moe_tile_bound(N, E, bm) * 16, 4,
              al(-(-N // 1024) * E * 4), T * 4, N * I * 4, N * H * 4]
    if Is:
        tables += [T * Is * 4, T * H * 4]
    assert _workspace(T, H, E, I, Is, k, logits_given) == sum(al(b) for b in tables)


def test_bf16_plan_rejects_bad_sizes():
    out = (ctypes.c_int * 4)()
    assert _lib.lib().sllm_moe_bf16_plan_query(4, 100, 8, 128, 0, 2, 1, out) == -1
    assert _lib.lib().sllm_moe_bf16_plan_query(4, 256, 8, 128, 0, 9, 1, out) == -1


GEMV, TILED = 5, 6


def _linear(fp4, M, N, K, bh=128, bw=None, aligned=1):
    return _lib.lib().sllm_linear_plan_query(fp4, M, N, K, bh, bw or (32 if fp4 else 128), aligned)


# rows that stream through the GEMV, rows from which the matrix cores run
@pytest.mark.parametrize("fp4,N,K,gemv,wide", [
    (0, 4096, 4096, (1, 2), (3, 64, 65)), (0, 7168, 2048, (2, 3), (4,)), (0, 2048, 7168, (1,), (2,)),
    (0, 256, 256, (1,), (2,)), (0, 12288, 4096, (2, 4), (5,)), (0, 14336, 4096, (1,), (2,)),
    (0, 17408, 5120, (2, 3), (4,)), (0, 151936, 2048, (2,), (3,)),
    (1, 4096, 4096, (1, 2), (3,)), (1, 2048, 2048, (2, 3), (4,)), (1, 2048, 7168, (1,), (2,)),
    (1, 256, 256, (1,), (2,)), (1, 18432, 7168, (2,), (3,)), (1, 20480, 2048, (2, 4), (5,)),
    (1, 32000, 4096, (1,), (2,))])
def test_linear_few_rows(fp4, N, K, gemv, wide):
    for M in gemv:
        assert _linear(fp4, M, N, K) == GEMV, M
    for M in wide:
        assert 0 <= _linear(fp4, M, N, K) < GEMV, M


def test_fp8_tile_by_rounds():
    """4096 columns: 32 x 256 tiles for a full round and an even number of
    them, 32 x 128 in between."""
    for M, tile in ((16, 0), (32, 1), (128, 2), (256, 3), (300, 4), (512, 4), (513, 3), (768, 3),
                    (1000, 4), (1024, 4)):
        assert _linear(0, M, 4096, 4096) == tile, M


def test_linear_fallbacks():
    """What the matrix-core kernel does not take: unaligned operands, a K
    that is no multiple of 64, other scale blocks."""
    assert _linear(0, 8, 256, 256, aligned=0) == GEMV
    assert _linear(0, 80, 256, 256, aligned=0) == TILED
    assert _linear(0, 8, 300, 200) == TILED        # ragged for both
    assert _linear(0, 8, 256, 256, bh=6) == TILED  # block rows not in fours
    assert _linear(0, 8, 256, 256, bw=192) == TILED
    assert 0 <= _linear(0, 8, 256, 256, bh=4, bw=64) < GEMV
    assert _linear(0, 1, 300, 256) == TILED        # one row off the 128 grid
    assert _linear(1, 8, 256, 96) == GEMV
    assert _linear(1, 80, 256, 96) == TILED
    assert _linear(1, 8, 250, 96) == TILED
    assert _linear(1, 2, 250, 256) < GEMV
    assert _linear(1, 8, 256, 256, bw=16) == TILED
    assert _linear(0, 0, 256, 256) == -1


@pytest.mark.parametrize("hole", [0, 1, 2, 3])
def test_linears_refuse_null_pointers(hole):
    """Before any launch, at every batch size."""
    lib = _lib.lib()
    for M in (1, 8, 80):
        p = [ctypes.c_void_p(0 if i == hole else 4096) for i in range(4)]
        assert lib.sllm_fp8_gemm_dev(*p, M, 128, 128, 128, 128) == -1
        assert "null" in _lib.last_error()
        assert lib.sllm_ds_fp4_gemm_packed_dev(*p, M, 128, 128, 32) == -1
        assert "null" in _lib.last_error()
