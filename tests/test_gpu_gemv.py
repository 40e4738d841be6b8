"""The unpacked-weight GEMV (decode.hip): every output of a wave's 4 x 4 sums
against the fp64 product, over rows short of four and K short of a wave's
lanes.

Bound. A lane rounds each product's addition in chains of C values and the
chains once each (c of them to a lane); the wave's sum is in 64 bits, with one
rounding at its end; an FP8 weight times its scale is rounded once:
|error| <= (C + c + 3) 2^-24 sum |a w|."""
import numpy as np
import pytest

from oracle import codecs

pytestmark = pytest.mark.gpu


def _check(got, a, wd, chain, lane_values):
    K = a.shape[1]
    want = a.astype(np.float64) @ wd.astype(np.float64).T
    mag = np.abs(a).astype(np.float64) @ np.abs(wd).astype(np.float64).T
    bound = (chain + 2 * -(-K // (64 * lane_values)) + 3) * 2.0 ** -24 * mag
    assert np.all(np.abs(got - want) <= bound), np.max(np.abs(got - want) / mag) * 2 ** 24


@pytest.mark.parametrize("M", [1, 2, 3, 4, 7, 64])
@pytest.mark.parametrize("N,K", [(16, 4), (48, 252), (160, 260), (32, 2048)])
def test_fp32_rows(M, N, K):
    from sllm_amd import q4
    rng = np.random.default_rng(M * N + K)
    a = rng.standard_normal((M, K)).astype(np.float32)
    w = rng.standard_normal((N, K)).astype(np.float32)
    _check(q4.gemv_rows(a, w, 0, 1.0), a, w, 4, 4)


@pytest.mark.parametrize("M,N,K", [(1, 128, 128), (1, 384, 1152), (2, 128, 2048), (3, 256, 2048),
                                   (4, 9216, 1024), (4, 20480, 1024)])
def test_quantized_few_rows(M, N, K):
    from sllm_amd import _lib, deepseek, fp8
    rng = np.random.default_rng(N + K)
    gemv = [_lib.lib().sllm_linear_plan_query(f, M, N, K, 128, 32 if f else 128, 1) == 5
            for f in (0, 1)]
    assert any(gemv)
    a = rng.standard_normal((M, K)).astype(np.float32)
    q = rng.integers(0, 256, (N, K), dtype=np.uint8)
    q[(q & 0x7F) == 0x7F] = 0x30
    s = (rng.random((N // 128, K // 128)) + 0.5).astype(np.float32)
    if gemv[0]:
        _check(fp8.fp8_gemm(a, q, s), a, codecs.dequant_fp8_block(q, s), 16, 16)
    p = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
    sc = rng.integers(115, 130, (N, K // 32), dtype=np.uint8)
    if gemv[1]:
        _check(deepseek.fp4_moe_linear(a, p, sc), a, codecs.dequant_fp4_block(p, sc), 16, 32)
