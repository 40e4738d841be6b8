"""The prompts' two routers, on both sides of the rule that picks one
(router.hip router_short: at most 32 tiles of 64 tokens x 128 experts): the
split small-batch router with full-row routing, its K slices in the y rows,
and the fused router. Logits against fp64, ids exact against the oracle on
those logits, the call without a logits copy bit for bit the call with one,
outputs against the call given the logits."""
import numpy as np
import pytest

from tests._fixtures import (check_qwen_routing, check_router_logits, deepseek_layer,
                             deepseek_mxfp4_gpu, qwen_fp8_gpu, qwen_layer, rel_l2)

pytestmark = pytest.mark.gpu


# short: one K chunk (H 512), two (2048), three (2304), ragged token tiles and
# expert tiles, every chunk-histogram size; then more than 32 tiles
@pytest.mark.parametrize("T,E,k,H", [
    (65, 16, 4, 512), (128, 64, 6, 2048), (190, 129, 4, 2304), (511, 512, 10, 2048),
    (2048, 64, 2, 512),
    (513, 512, 10, 512), (2100, 96, 16, 512), (1030, 200, 8, 512), (330, 1024, 10, 512),
    (140, 2048, 10, 512), (2049, 129, 1, 512)])
def test_qwen_prompt_routers(T, E, k, H):
    x, W = qwen_fp8_gpu(seed=T + E, T=T, H=H, E=E, I=128, Is=128)
    layer = qwen_layer(W, k)
    y, r = layer.forward(x, mode="prefill", return_routing=True)
    check_router_logits(f"T={T} E={E} H={H}", x, W.router_w, r["logits"])
    check_qwen_routing(r["logits"], r["ids"], r["w"], k)
    np.testing.assert_array_equal(r["counts"], np.bincount(r["ids"].ravel(), minlength=E))
    y_g, r_g = layer.forward(x, logits=r["logits"], mode="prefill", return_routing=True)
    np.testing.assert_array_equal(r["ids"], r_g["ids"])
    # the same rows and weights (to the normaliser's order) through bf16 y rows
    assert rel_l2(y, y_g) < 1e-4
    np.testing.assert_array_equal(layer.forward(x, mode="prefill"), y)


@pytest.mark.parametrize("T,H", [(65, 2304), (200, 512), (70, 7168)])
def test_deepseek_short_prompt_router(T, H):
    x, W = deepseek_mxfp4_gpu(seed=T, T=T, H=H, E=32, I=256, Is=256)
    layer = deepseek_layer(W, 4, n_group=4, topk_group=2, route_scale=2.5, swiglu_limit=10.0)
    y, r = layer.forward(x, mode="prefill", return_routing=True)
    check_router_logits(f"DeepSeek T={T} H={H}", x, W.router_w, r["logits"])
    y_g, r_g = layer.forward(x, logits=r["logits"], mode="prefill", return_routing=True)
    # the slices' sum is what the logits copy holds: the same routing, rows
    # and sums, bit for bit
    np.testing.assert_array_equal(r["ids"], r_g["ids"])
    np.testing.assert_array_equal(r["w"], r_g["w"])
    np.testing.assert_array_equal(y, y_g)
    np.testing.assert_array_equal(layer.forward(x, mode="prefill"), y)


# bf16 gemm_ex above 64 rows: the K-split kernel (a few 64 x 128 tiles, K from
# 640; one to four slices a wave, a partial round), the tiles at shorter K, at
# many rows with K 1280, and past 32 tiles
@pytest.mark.parametrize("m,n,k", [
    (65, 200, 640), (300, 129, 1024), (1290, 100, 1152), (70, 2000, 1792), (2048, 16, 1408),
    (300, 129, 512), (1290, 100, 1280), (2049, 70, 1664), (330, 770, 1024)])
def test_bf16_gemm_both_kernels(m, n, k):
    """Products of bf16 values are exact in fp32; each of the K / 32 MFMA
    steps adds 32 of them with a few roundings, the K-split kernel's waves
    once more: |error| <= (K / 32 * 6 + 8) 2^-24 sum |a w|."""
    from oracle import codecs
    from sllm_amd.runtime import DeviceBuffer, T_BF16, gemm_ex, sync, to_bf16, to_device_raw
    rng = np.random.default_rng(m * n + k)
    a = codecs.round_bf16(rng.standard_normal((m, k)).astype(np.float32))
    w = codecs.round_bf16(rng.standard_normal((n, k)).astype(np.float32))
    c = DeviceBuffer(m * n * 4)
    gemm_ex(to_device_raw(to_bf16(a)), to_device_raw(to_bf16(w)), c, m, n, k, T_BF16)
    sync()
    want = a.astype(np.float64) @ w.astype(np.float64).T
    mag = np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64).T
    assert np.all(np.abs(c.copy_host().reshape(m, n) - want) <= (k / 32 * 6 + 8) * 2.0 ** -24 * mag)
