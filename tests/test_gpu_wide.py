"""The matrix-core kernel over unpacked weights (gemm_wide.hip) at the edges
of its tiles: FP8 and MXFP4 linears against the fp64 product, the bf16 layer
against the reference's per-token loop, non-finite activations and scales.

Bound. Every product is exact (an fp32 activation as three bf16 parts); a
64-wide K step adds at most 6 rounded MFMA sums and one rounded add, and the
K waves' sums up to 8 more, so |error| <= (7 ceil(K / 64) + 8) 2^-24 sum |a w|,
plus one rounding of each FP8 scale product."""
import numpy as np
import pytest

from oracle import codecs
from oracle import qwen_moe as qm

pytestmark = pytest.mark.gpu

bf = codecs.round_bf16


def _check(got, a, wd):
    want = a.astype(np.float64) @ wd.astype(np.float64).T
    mag = np.abs(a).astype(np.float64) @ np.abs(wd).astype(np.float64).T
    K = a.shape[1]
    bound = (8 * -(-K // 64) + 8) * 2.0 ** -24 * mag + 1e-30
    assert np.all(np.abs(got - want) <= bound), np.max(np.abs(got - want) / bound)


# rows at the tiles' edges; columns short of a tile, a scale block or a
# 16-column subtile; K of one step, of a partial last step over the K waves
@pytest.mark.parametrize("M", [2, 16, 17, 33, 65, 130])
@pytest.mark.parametrize("N,K,bh,bw", [(128, 128, 128, 128), (576, 192, 128, 128),
                                       (133, 64, 4, 64), (40, 1088, 64, 256),
                                       (2112, 512, 128, 128)])
def test_fp8_linear(M, N, K, bh, bw):
    from sllm_amd import fp8
    rng = np.random.default_rng(M * N + K)
    a = (rng.standard_normal((M, K)) * 10.0 ** rng.integers(-3, 4, (M, 1))).astype(np.float32)
    q = rng.integers(0, 256, (N, K), dtype=np.uint8)
    q[(q & 0x7F) == 0x7F] = 0x30
    s = (rng.random((-(-N // bh), -(-K // bw))) + 0.5).astype(np.float32)
    _check(fp8.fp8_gemm(a, q, s, bh, bw), a, codecs.dequant_fp8_block(q, s, (bh, bw)))


@pytest.mark.parametrize("M", [2, 17, 65])
@pytest.mark.parametrize("N,K", [(16, 64), (200, 320), (2048, 1088)])
def test_fp4_linear(M, N, K):
    from sllm_amd import deepseek
    rng = np.random.default_rng(M + N * K)
    a = rng.standard_normal((M, K)).astype(np.float32)
    p = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
    s = rng.integers(115, 130, (N, K // 32), dtype=np.uint8)
    s[0, 0] = 0  # a zero scale
    _check(deepseek.fp4_moe_linear(a, p, s), a, codecs.dequant_fp4_block(p, s))


# each tile (16 x 16, 16 x 32, 32 x 64, 32 x 128, FP8 32 x 256 or MXFP4 64 x
# 128) with ragged rows and columns; K of one step, a partial last step over
# the K waves, more than the four steps of the unrolled loop
@pytest.mark.parametrize("fp4", [0, 1])
@pytest.mark.parametrize("tile,M,N", [(0, 10, 520), (1, 30, 4090), (2, 35, 4090), (3, 200, 4090),
                                      (4, 500, 4090)])
@pytest.mark.parametrize("K", [64, 320, 1088])
def test_every_linear_tile(fp4, tile, M, N, K):
    from sllm_amd import _lib, deepseek, fp8
    assert _lib.lib().sllm_linear_plan_query(fp4, M, N, K, 128, 32 if fp4 else 128, 1) == tile
    rng = np.random.default_rng(tile + K)
    a = rng.standard_normal((M, K)).astype(np.float32)
    if fp4:
        p = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
        s = rng.integers(115, 130, (N, K // 32), dtype=np.uint8)
        _check(deepseek.fp4_moe_linear(a, p, s), a, codecs.dequant_fp4_block(p, s))
    else:
        q = rng.integers(0, 0x70, (N, K), dtype=np.uint8)
        s = (rng.random((-(-N // 128), -(-K // 128))) + 0.5).astype(np.float32)
        _check(fp8.fp8_gemm(a, q, s), a, codecs.dequant_fp8_block(q, s))


@pytest.mark.parametrize("M", [3, 40])
def test_nonfinite_activations(M):
    """An infinite activation gives its row's outputs the infinity of its
    weight's sign, a NaN gives NaN; the other rows and the largest finite
    value are as without them. A NaN scale gives its output column NaN."""
    from sllm_amd import deepseek, fp8
    rng = np.random.default_rng(M)
    N, K = 96, 256
    a = rng.standard_normal((M, K)).astype(np.float32)
    a[0, 5], a[1, 7], a[2, 9] = np.inf, np.nan, np.finfo(np.float32).max
    q = rng.integers(0x20, 0x30, (N, K), dtype=np.uint8)
    q[::3] |= 0x80
    s = np.ones((1, 2), np.float32)
    got = fp8.fp8_gemm(a, q, s)
    wd = codecs.dequant_fp8_block(q, s)
    np.testing.assert_array_equal(got[0], np.where(wd[:, 5] > 0, np.inf, -np.inf))
    assert np.all(np.isnan(got[1]))
    _check(got[2:], a[2:], wd)
    p = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
    sc = np.full((N, K // 32), 127, np.uint8)
    sc[4, 1] = 255
    y = deepseek.fp4_moe_linear(rng.standard_normal((M, K)).astype(np.float32), p, sc)
    assert np.all(np.isnan(y[:, 4]))
    assert np.all(np.isfinite(np.delete(y, 4, 1)))


def test_nonfinite_rows_of_a_tall_tile():
    """NaN, infinite and overflowing rows of one 32-row tile beside each
    other: each row as a plain product has it, the finite ones untouched."""
    from sllm_amd import _lib, fp8
    M, N, K = 500, 4090, 128
    assert _lib.lib().sllm_linear_plan_query(0, M, N, K, 128, 128, 1) == 4
    rng = np.random.default_rng(7)
    a = rng.standard_normal((M, K)).astype(np.float32)
    q = rng.integers(0x20, 0x70, (N, K), dtype=np.uint8)
    q[::3] |= 0x80
    q[5, 9] = 0
    s = np.full((-(-N // 128), 1), 1e-3, np.float32)
    clean = fp8.fp8_gemm(a, q, s)
    a[3, 7], a[19, 100], a[35, 9], a[50] = np.nan, np.inf, -np.inf, 3e37
    a[51, 0], a[51, 1] = np.inf, -np.inf
    got = fp8.fp8_gemm(a, q, s)
    wd = codecs.dequant_fp8_block(q, s)
    for m in (3, 19, 35, 51):
        np.testing.assert_array_equal(got[m], _product(a[m:m + 1], wd)[0])
    _check(got[50:51], a[50:51], wd)
    keep = np.setdiff1d(np.arange(M), (3, 19, 35, 50, 51))
    np.testing.assert_array_equal(got[keep], clean[keep])


def test_every_pair_of_fp8_codes():
    """One-hot activations read the converted weights back: every pair of
    finite codes, in either half of a dword, exactly."""
    from sllm_amd import fp8
    K, N = 64, 2048
    codes = np.arange(65536, dtype=np.uint32)
    q = np.stack([codes & 255, codes >> 8], -1).astype(np.uint8)
    q[(q & 0x7F) == 0x7F] = 0
    for q2 in (q, np.roll(q, 1, axis=0)):  # (each pair in the other half)
        w = q2.reshape(N, K)
        got = fp8.fp8_gemm(np.eye(K, dtype=np.float32), w, np.ones((N // 128, 1), np.float32),
                           128, 64)
        np.testing.assert_array_equal(got, codecs.decode_e4m3fn(w).T)


def _product(a, wd):
    """The fp64 product with what 0 and infinities give (an fp32 overflow as
    an infinity)."""
    with np.errstate(all="ignore"):
        return (a.astype(np.float64)[:, None, :] * wd.astype(np.float64)[None]).sum(-1) \
            .astype(np.float32)


@pytest.mark.parametrize("M", [3, 40, 260])
def test_fp8_linear_block_scale_range(M):
    """Activations whose products with the unscaled codes overflow: the block
    scale belongs to the weight, so a small one keeps the result finite, a
    zero one makes it 0, an infinite one infinite (NaN beside a zero code)."""
    from sllm_amd import fp8
    rng = np.random.default_rng(M)
    N, K = 520, 256
    a = (rng.standard_normal((M, K)) + 2.0).astype(np.float32) * np.float32(1e36)
    a[1] = 1.0  # exact in bf16: nothing in its two lower parts
    q = rng.integers(0x70, 0x7F, (N, K), dtype=np.uint8)
    q[::2, ::3] |= 0x80
    s = np.full((5, 2), 1e-3, np.float32)
    s[1] = 0.0
    s[2, 1] = np.inf
    q[260:300, 130] = 0
    got = fp8.fp8_gemm(a, q, s)
    wd = codecs.dequant_fp8_block(q, s)
    finite = np.r_[0:256, 384:N]
    _check(got[:, finite], a, wd[finite])
    assert np.all(got[:, 128:256] == 0)
    np.testing.assert_array_equal(got[:, 256:384], _product(a, wd[256:384]))


@pytest.mark.parametrize("M", [3, 40])
@pytest.mark.parametrize("e", [-112, -124, -136])
def test_tiny_activations(M, e):
    """Activations near and below fp32's smallest normal value keep their
    bits: the result is a plain fp32 product's to its rounding."""
    from sllm_amd import deepseek, fp8
    rng = np.random.default_rng(M - e)
    N, K = 96, 256
    a = np.ldexp(rng.standard_normal((M, K)), e).astype(np.float32)
    q = rng.integers(0, 0x70, (N, K), dtype=np.uint8)
    s = np.full((1, 2), 2.0 ** 60, np.float32)
    p = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
    sc = np.full((N, K // 32), 127 + 60, np.uint8)
    for got, wd in ((fp8.fp8_gemm(a, q, s), codecs.dequant_fp8_block(q, s)),
                    (deepseek.fp4_moe_linear(a, p, sc), codecs.dequant_fp4_block(p, sc))):
        mag = np.abs(a).astype(np.float64) @ np.abs(wd).astype(np.float64).T
        err = np.abs(got - a.astype(np.float64) @ wd.astype(np.float64).T)
        assert np.all(err <= (8 * (K // 64) + 8) * 2.0 ** -24 * mag), np.max(err / mag)


@pytest.mark.parametrize("M", [2, 40])
def test_infinite_weights(M):
    """An infinite weight (e8m0 254; a bf16 one in the down projection) gives
    its outputs the infinity of the product's sign, as a plain product does,
    also where the activation is exact in bf16."""
    from sllm_amd import deepseek
    from sllm_amd.moe import QwenMoE
    rng = np.random.default_rng(M)
    N, K = 48, 128
    a = rng.integers(1, 5, (M, K)).astype(np.float32)
    p = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
    p[:, 16:32] = 0
    p[:, 16] = 0x44  # twice 2, times 2^127 where the scale is 254
    s = np.full((N, K // 32), 127, np.uint8)
    s[::2, 1] = 254
    got = deepseek.fp4_moe_linear(a, p, s)
    assert np.all(np.isposinf(got[:, ::2]))
    _check(got[:, 1::2], a, codecs.dequant_fp4_block(p, s)[1::2])

    E, I, H, T = 2, 128, 256, 3 * M
    w = lambda *n: bf((rng.standard_normal(n) * 0.05).astype(np.float32))  # noqa: E731
    x, rw, wg, wu, wd = bf(rng.standard_normal((T, H)).astype(np.float32)), w(E, H), \
        w(E, I, H), w(E, I, H), w(E, H, I)
    wu[:, 5] = 0  # h = 0 there: NaN against an infinite weight
    wd[0, 7, 9], wd[1, 11, 3], wd[0, 20, 5] = np.inf, -np.inf, np.inf
    logits = rng.standard_normal((T, E)).astype(np.float32)
    got = QwenMoE(rw, wg, wu, wd, top_k=1).forward(x, logits=logits)
    with np.errstate(all="ignore"):
        want = qm.moe_block_grouped(x, logits, wg, wu, wd, 1, None)
    fin = np.isfinite(want)
    np.testing.assert_array_equal(got[~fin], want[~fin])
    np.testing.assert_allclose(got[fin], want[fin], rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("T,k,shared,H", [
    (1, 2, True, 256), (5, 3, False, 256), (33, 2, True, 256), (70, 4, True, 256),
    (260, 1, False, 256), (2900, 3, True, 256), (1701, 5, False, 256),
    (90, 2, True, 2048), (200, 3, True, 1280)])
def test_bf16_layer_tiles(T, k, shared, H):
    """Each tile of the bf16 layer (by assignments: 16-row, 32 x 64, 32 x
    128, 64 x 256), a ragged last row tile, empty experts, with and without the shared
    segment, against the per-token loop (fp32 there too). Above 64 tokens the
    router's launch also forms the shared gate: in one K chunk, or (H 1280,
    2048) in two partials."""
    from sllm_amd.moe import QwenMoE
    rng = np.random.default_rng(T)
    E, I, Is = 6, 128, 256

    def w(*shape):
        return bf((rng.standard_normal(shape) * 0.05).astype(np.float32))
    x = bf(rng.standard_normal((T, H)).astype(np.float32))
    rw, wg, wu, wd = w(E, H), w(E, I, H), w(E, I, H), w(E, H, I)
    sg, su, sd, sgl = (w(Is, H), w(Is, H), w(H, Is), w(1, H)) if shared else (None,) * 4
    layer = QwenMoE(rw, wg, wu, wd, sg=sg, su=su, sd=sd, sgl=sgl, top_k=k)
    got, r = layer.forward(x, return_routing=True)
    want = qm.moe_block_grouped(x, r["logits"], wg, wu, wd, k,
                                (sg, su, sd, sgl) if shared else None)
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    # two chained fp32 products: a few 2^-24 each, the reference's own included
    assert rel < 2e-6, rel


# with a shared expert on the GEMV (1, 2 tokens), the 16-row tiles and the
# 32-row ones; above 64 tokens (the router's launch split); without a shared
# expert
@pytest.mark.parametrize("T,E,k,shared,H,I", [
    (1, 24, 4, True, 2048, 1408), (2, 24, 4, True, 2048, 1408), (3, 24, 4, True, 2048, 1408),
    (10, 24, 4, True, 2048, 1408), (20, 64, 5, True, 1280, 512), (70, 80, 2, True, 2048, 256),
    (7, 16, 2, False, 256, 128), (80, 64, 2, False, 1280, 128),
    (2, 1, 1, False, 512, 256)])
def test_bf16_layer_few_rows(T, E, k, shared, H, I):
    """Few rows an expert: the routed GEMV with each kernel of the shared
    expert, against the per-token loop."""
    from sllm_amd.moe import QwenMoE
    rng = np.random.default_rng(T + E)
    Is = 384

    def w(*shape):
        return bf(rng.standard_normal(shape, dtype=np.float32) * np.float32(0.05))
    x = bf(rng.standard_normal((T, H)).astype(np.float32))
    rw, wg, wu, wd = w(E, H), w(E, I, H), w(E, I, H), w(E, H, I)
    sg, su, sd, sgl = (w(Is, H), w(Is, H), w(H, Is), w(1, H)) if shared else (None,) * 4
    layer = QwenMoE(rw, wg, wu, wd, sg=sg, su=su, sd=sd, sgl=sgl, top_k=k)
    got, r = layer.forward(x, return_routing=True)
    want = qm.moe_block_grouped(x, r["logits"], wg, wu, wd, k,
                                (sg, su, sd, sgl) if shared else None)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < 2e-6


def _off(a, by=8):
    """A device copy of `a` that begins `by` bytes past an aligned address."""
    from sllm_amd.runtime import to_device_raw
    raw = np.ascontiguousarray(a).view(np.uint8).reshape(-1)
    buf = to_device_raw(np.concatenate([np.zeros(by, np.uint8), raw]))
    return buf, buf.ptr + by


# rows an expert below and above 16, below and above a 64-row tile
@pytest.mark.parametrize("T,k,shared", [(3, 2, True), (40, 2, False), (90, 2, True), (300, 3, True)])
def test_bf16_layer_unaligned_weights(T, k, shared):
    """Weights 8 bytes past a 16-byte boundary: the GEMV, against the
    per-token loop."""
    import ctypes
    from sllm_amd import _lib
    from sllm_amd.moe import qwen_workspace_bytes
    from sllm_amd.runtime import DeviceBuffer, sync, to_bf16, to_device_raw
    rng = np.random.default_rng(T)
    H, E, I = 256, 5, 128

    def w(*shape):
        return bf((rng.standard_normal(shape) * 0.05).astype(np.float32))
    x = bf(rng.standard_normal((T, H)).astype(np.float32))
    W = dict(router_w=w(E, H), wg=w(E, I, H), wu=w(E, I, H), wd=w(E, H, I))
    if shared:
        W.update(sg=w(I, H), su=w(I, H), sd=w(H, I), sgl=w(1, H))
    logits = DeviceBuffer(T * E * 4)
    out = DeviceBuffer(T * H * 4)
    nb = qwen_workspace_bytes(T, H, E, I, I if shared else 0, k, has_shared=shared, wdtype=1)
    ws, xb = DeviceBuffer(nb), to_device_raw(to_bf16(x))
    a = _lib.QwenArgs()
    a.T, a.H, a.E, a.I, a.Is, a.topk = T, H, E, I, I if shared else 0, k
    a.out_f32, a.wdtype, a.renorm_eps = 1, 1, 1e-20
    a.x, a.out, a.logits_out, a.workspace, a.workspace_bytes = xb.ptr, out.ptr, logits.ptr, ws.ptr, nb
    keep = {}
    for name, v in W.items():
        buf, p = _off(to_bf16(v), 0 if name in ("router_w", "sgl") else 8)
        keep[name] = buf
        setattr(a, name, p)
    _lib.check(_lib.lib().sllm_moe_qwen_forward(ctypes.byref(a)), "qwen")
    sync()
    want = qm.moe_block_grouped(x, logits.copy_host().reshape(T, E), W["wg"], W["wu"], W["wd"], k,
                                (W["sg"], W["su"], W["sd"], W["sgl"]) if shared else None)
    got = out.copy_host().reshape(T, H)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < 2e-6


@pytest.mark.parametrize("M", [2, 40, 70])
def test_unaligned_linears(M):
    """FP8 and MXFP4 weights 8 bytes past a 16-byte boundary, and FP8
    activations 4 past: the GEMV up to 64 rows, the tiled kernel above."""
    from sllm_amd import deepseek, fp8
    from sllm_amd.runtime import DeviceBuffer, sync
    rng = np.random.default_rng(M)
    N, K = 128, 256
    a = rng.standard_normal((M, K)).astype(np.float32)
    q = rng.integers(0, 0x70, (N, K), dtype=np.uint8)
    s = (rng.random((1, 2)) + 0.5).astype(np.float32)
    p = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
    sc = rng.integers(115, 130, (N, K // 32), dtype=np.uint8)
    out = DeviceBuffer(M * N * 4)
    bufs = [_off(a, 0), _off(q), _off(s, 0), _off(a, 4), _off(p), _off(sc, 0)]
    d = [b[1] for b in bufs]

    def check(wd):
        sync()
        got = out.copy_host().reshape(M, N)
        # the tiled kernel adds K products one by one: (K + 2) 2^-24
        mag = np.abs(a).astype(np.float64) @ np.abs(wd).astype(np.float64).T
        err = np.abs(got - a.astype(np.float64) @ wd.astype(np.float64).T)
        assert np.all(err <= (K + 2) * 2.0 ** -24 * mag)
    fp8.fp8_gemm_dev(d[0], d[1], d[2], out, M, N, K)
    check(codecs.dequant_fp8_block(q, s))
    fp8.fp8_gemm_dev(d[3], d[1], d[2], out, M, N, K)
    check(codecs.dequant_fp8_block(q, s))
    deepseek.fp4_moe_linear_dev(d[0], d[4], d[5], out, M, N, K)
    check(codecs.dequant_fp4_block(p, sc))


@pytest.mark.parametrize("T", [3, 40])
def test_bf16_layer_infinity(T):
    """An infinite activation under positive weights leaves its token
    infinite, not NaN through the compensated sum; the others as without."""
    from sllm_amd.moe import QwenMoE
    rng = np.random.default_rng(T)
    E, I, H, k = 4, 128, 1024, 2

    def w(*shape):
        return bf((rng.random(shape) * 0.05 + 0.01).astype(np.float32))
    x = bf(rng.standard_normal((T, H)).astype(np.float32))
    logits = rng.standard_normal((T, E)).astype(np.float32)
    layer = QwenMoE(w(E, H), w(E, I, H), w(E, I, H), w(E, H, I), top_k=k)
    want = layer.forward(x, logits=logits)
    x[0, 5] = np.inf
    got = layer.forward(x, logits=logits)
    assert np.all(got[0] == np.inf)
    np.testing.assert_array_equal(got[1:], want[1:])
