"""The work that users of this library have it do, as timed cases.

A case is a dict of plain values. `listed()` gives the named ones, `draw(rng)`
another one of the same ranges, `prepare(case, seed)` what a serving program
holds before the call (weights resident and packed on the GPU, activations,
output and workspace), `run(state)` one pass through the public entry points,
`exact(case, seed)` the same values in 64 bits by plain torch, `work(case)`
the bytes and operations that a pass cannot do without, and
`tolerance(case)` how far two correct implementations may be apart.

Kinds of case:
  qwen    the Qwen-style FP8 MoE layer (softmax top-k, gated shared expert):
          decode batches through DeviceMoEStack.moe_dev (fp32 result), prompts
          through qwen_forward_dev (bf16 result), `skew` with a routing bias
  ds      the DeepSeek-style layer (sigmoid group-limited routing, MXFP4
          experts, FP8 shared expert) through deepseek_forward_dev
  bf16    the Qwen-style layer with bf16 weights (the precision of
          moe_block_forward and of DeviceMoEStack.from_weights)
  dense   a dense FP8 SwiGLU MLP through DenseSwiGLU.forward_dev
  fp8     the FP8 block-scaled linear, fp8_gemm_dev
  fp4     the MXFP4 linear, fp4_moe_linear_dev

torch comes first, so that the library and torch share one HIP runtime.
"""

import torch

from sllm_amd import fp8 as _fp8
from sllm_amd import moe as _moe
from sllm_amd import deepseek as _ds
from sllm_amd.decode import DenseSwiGLU, DeviceMoEStack

GPU = "cuda:0"

# layer geometries: hidden, experts, intermediate, shared intermediate, top-k
QWEN = {"H": 2048, "E": 512, "I": 512, "Is": 512, "k": 10}
DEEPSEEK = {"H": 7168, "E": 256, "I": 2048, "Is": 2048, "k": 8}
SMALL = {"H": 1024, "E": 16, "I": 512, "Is": 512, "k": 4}
# groups, kept groups, routed scaling and SwiGLU clamp of the DeepSeek layer
N_GROUP, TOPK_GROUP, ROUTE_SCALE, LIMIT = 8, 4, 2.5, 10.0
# the skewed prompts: bias -SKEW ln(rank), which gives the top tenth of the
# experts about 60% of the assignments; the last twentieth stays empty
SKEW = 0.42


def listed():
    return [
        # one user's decode step: launches and latency
        {"name": "decode_1", "kind": "qwen", "T": 1, "skew": False, **QWEN},
        # a serving batch's decode step
        {"name": "decode_32", "kind": "qwen", "T": 32, "skew": False, **QWEN},
        # one short prompt of a ragged length
        {"name": "prompt_333", "kind": "qwen", "T": 333, "skew": False, **QWEN},
        # a prefill chunk
        {"name": "prefill_4096", "kind": "qwen", "T": 4096, "skew": False, **QWEN},
        # the largest chunk, with hot and empty experts
        {"name": "prefill_16384_skew", "kind": "qwen", "T": 16384, "skew": True, **QWEN},
        # the large layer's decode step for a small batch
        {"name": "ds_decode_8", "kind": "ds", "T": 8, **DEEPSEEK},
        # the large layer's prefill chunk
        {"name": "ds_prefill_8192", "kind": "ds", "T": 8192, **DEEPSEEK},
        # the small model in bf16: a decode batch, and a prompt
        {"name": "bf16_64", "kind": "bf16", "T": 64, **SMALL},
        {"name": "bf16_prompt_1000", "kind": "bf16", "T": 1000, **SMALL},
        # a dense model's MLP in a decode step
        {"name": "dense_mlp_8", "kind": "dense", "T": 8, "H": 5120, "I": 17408},
        # a projection of an FP8 checkpoint over a prompt
        {"name": "fp8_linear_512", "kind": "fp8", "T": 512, "N": 4096, "K": 4096},
        # one expert's MXFP4 projection over the tokens routed to it
        {"name": "fp4_linear_300", "kind": "fp4", "T": 300, "N": 2048, "K": 7168},
    ]


def _log(rng, lo, hi):
    """A whole number, spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    case = _drawn(rng)
    while case in [{k: v for k, v in c.items() if k != "name"} for c in listed()]:
        case["T"] += -1 if case["T"] > 1 else 1
    return case


def _drawn(rng):
    kind = rng.choice(["qwen", "qwen", "qwen", "ds", "bf16", "dense", "fp8", "fp4"])
    if kind == "qwen":
        geo = rng.choice([
            QWEN,
            {"H": 2048, "E": 128, "I": 768, "Is": 0, "k": 8},
            {"H": 3072, "E": 64, "I": 1408, "Is": 1408, "k": 6},
        ])
        T = _log(rng, 1, 16384)
        return {"kind": kind, "T": T, "skew": T > 512 and rng.random() < 0.3, **geo}
    if kind == "ds":
        return {"kind": kind, "T": _log(rng, 1, 8191), **DEEPSEEK}
    if kind == "bf16":
        geo = rng.choice([SMALL, {"H": 2048, "E": 32, "I": 768, "Is": 0, "k": 4}])
        return {"kind": kind, "T": _log(rng, 1, 999), **geo}
    if kind == "dense":
        H, I = rng.choice([(5120, 17408), (2048, 5632), (4096, 12288)])
        return {"kind": kind, "T": _log(rng, 1, 64), "H": H, "I": I}
    T = _log(rng, 1, 512)
    if kind == "fp8":  # projections, some with a ragged number of rows
        N, K = rng.choice([1536, 2048, 2112, 4096]), rng.choice([2048, 3072, 4096])
    else:
        N, K = rng.choice([(2048, 7168), (7168, 2048), (1536, 4096)])
    return {"kind": kind, "T": T, "N": N, "K": K}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=GPU)
    g.manual_seed(int(seed) % (1 << 62))
    return g


def _normal(g, *shape, std=1.0, dtype=torch.float32):
    return torch.randn(*shape, device=GPU, generator=g).mul_(std).to(dtype)


def _fp8_weight(g, rows, cols, pow2=False):
    """N(0, 0.02) in e4m3 with 128 x 128 block scales: codes, scales."""
    rb, cb = -(-rows // 128), -(-cols // 128)
    w = torch.zeros(rb * 128, cb * 128, device=GPU)
    w[:rows, :cols] = _normal(g, rows, cols, std=0.02)
    w = w.view(rb, 128, cb, 128)
    s = w.abs().amax(dim=(1, 3)) / 448.0
    if pow2:
        s = torch.exp2(torch.ceil(torch.log2(s)))
    q = (w / s[:, None, :, None]).to(torch.float8_e4m3fn)
    q = q.view(rb * 128, cb * 128)[:rows, :cols].contiguous()
    return q.view(torch.uint8), s.contiguous()


def _fp4_weight(g, rows, cols):
    """N(0, 0.02) in e2m1 (low nibble = even column) with an e8m0 scale for
    each 32 columns: packed codes, scales."""
    packed = torch.empty(rows, cols // 2, dtype=torch.uint8, device=GPU)
    scale = torch.empty(rows, cols // 32, dtype=torch.uint8, device=GPU)
    mid = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=GPU)
    step = max(1, (1 << 28) // cols)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        w = _normal(g, n, cols // 32, 32, std=0.02)
        e = torch.ceil(torch.log2(w.abs().amax(-1, keepdim=True) / 6.0))
        scale[r:r + n] = (e[..., 0] + 127).to(torch.uint8)
        w *= torch.exp2(-e)
        c = torch.bucketize(w.abs(), mid, out_int32=True).to(torch.uint8)
        c |= (w < 0).to(torch.uint8) << 3
        c = c.view(n, cols // 2, 2)
        packed[r:r + n] = c[..., 0] | (c[..., 1] << 4)
    return packed, scale


def _qwen_inputs(case, seed):
    g = _gen(seed)
    T, H, E, I, Is = case["T"], case["H"], case["E"], case["I"], case["Is"]
    w = {"router_w": _normal(g, E, H, std=0.02, dtype=torch.bfloat16)}
    if case["kind"] == "bf16":
        def put(name, *shape):
            w[name] = _normal(g, *shape, std=0.02, dtype=torch.bfloat16)
    else:
        def put(name, *shape):
            rows = 1
            for n in shape[:-1]:
                rows *= n
            w[name], w[name + "_s"] = _fp8_weight(g, rows, shape[-1])
    put("wg", E, I, H)
    put("wu", E, I, H)
    put("wd", E, H, I)
    if Is:
        put("sg", Is, H)
        put("su", Is, H)
        put("sd", H, Is)
        w["sgl"] = _normal(g, H, std=0.02, dtype=torch.bfloat16)
    if case.get("skew"):
        rank = torch.randperm(E, device=GPU, generator=g)
        w["router_bias"] = (-SKEW * torch.log(rank + 1.0)
                            - 64.0 * (rank >= E - E // 20)).float()
    x = _normal(g, T, H, dtype=torch.bfloat16)
    return w, x


def _ds_inputs(case, seed):
    g = _gen(seed)
    T, H, E, I, Is = case["T"], case["H"], case["E"], case["I"], case["Is"]
    w = {"router_w": _normal(g, E, H, std=0.02, dtype=torch.bfloat16),
         "bias": _normal(g, E, std=0.01)}
    w["w1"], w["w1_s"] = _fp4_weight(g, E * I, H)
    w["w3"], w["w3_s"] = _fp4_weight(g, E * I, H)
    w["w2"], w["w2_s"] = _fp4_weight(g, E * H, I)
    w["s1"], w["s1_s"] = _fp8_weight(g, Is, H, pow2=True)
    w["s3"], w["s3_s"] = _fp8_weight(g, Is, H, pow2=True)
    w["s2"], w["s2_s"] = _fp8_weight(g, H, Is, pow2=True)
    x = _normal(g, T, H, dtype=torch.bfloat16)
    return w, x


def _dense_inputs(case, seed):
    g = _gen(seed)
    T, H, I = case["T"], case["H"], case["I"]
    w = {"router_w": torch.zeros(1, H, dtype=torch.bfloat16, device=GPU)}
    w["wg"], w["wg_s"] = _fp8_weight(g, I, H)
    w["wu"], w["wu_s"] = _fp8_weight(g, I, H)
    w["wd"], w["wd_s"] = _fp8_weight(g, H, I)
    x = _normal(g, T, H, dtype=torch.bfloat16)
    return w, x


def _linear_inputs(case, seed):
    g = _gen(seed)
    make = _fp8_weight if case["kind"] == "fp8" else _fp4_weight
    w, s = make(g, case["N"], case["K"])
    return w, s, _normal(g, case["T"], case["K"])


def _decode(case):
    """The batches that the layer runs on unquantized activations."""
    return case["kind"] in ("bf16", "dense") or case["T"] <= 64


def _result(case):
    """Decode hooks return fp32, prompts bf16 as the next layer reads it."""
    dtype = torch.float32 if _decode(case) else torch.bfloat16
    return torch.empty(case["T"], case["H"], dtype=dtype, device=GPU)


def _sizes(case):
    return {"T": case["T"], "H": case["H"], "E": case["E"], "I": case["I"],
            "Is": case["Is"], "topk": case["k"]}


def _buffer(nbytes):
    return torch.empty(nbytes, dtype=torch.uint8, device=GPU)


def prepare(case, seed):
    kind, T = case["kind"], case["T"]
    state = {"case": case}
    if kind in ("fp8", "fp4"):
        state["w"], state["s"], state["x"] = _linear_inputs(case, seed)
        state["out"] = torch.empty(T, case["N"], device=GPU)
        return state
    H, I = case["H"], case["I"]
    if kind == "dense":
        w, state["x"] = _dense_inputs(case, seed)
        layer = _moe.QwenMoE.from_device(w, E=1, I=I, H=H, Is=0, top_k=1)
        state["mlp"] = DenseSwiGLU(layer)
    elif kind == "ds":
        w, state["x"] = _ds_inputs(case, seed)
        E, Is = case["E"], case["Is"]
        w["w13_packed"], w["w13_s_packed"] = _moe.pack_weights(
            1, 1, w["w1"], w["w3"], E, I, H, w["w1_s"], w["w3_s"])
        w["w2_packed"], w["w2_s_packed"] = _moe.pack_weights(
            1, 0, w["w2"], None, E, H, I, w["w2_s"])
        w["s13_packed"], _ = _moe.pack_weights(0, 1, w["s1"], w["s3"], 1, Is, H)
        w["s2_packed"], _ = _moe.pack_weights(0, 0, w["s2"], None, 1, H, Is)
        state["w"] = w
        state["ws"] = _buffer(_moe.deepseek_workspace_bytes(
            T, H, E, I, Is, case["k"]))
    else:
        w, state["x"] = _qwen_inputs(case, seed)
        E, Is = case["E"], case["Is"]
        if kind == "qwen":
            layer = _moe.QwenMoE.from_device(w, E=E, I=I, H=H, Is=Is,
                                             top_k=case["k"])
            w = layer._w  # with the packed copies
            if _decode(case):
                state["stack"] = DeviceMoEStack([layer])
        state["w"] = w
        state["ws"] = _buffer(_moe.qwen_workspace_bytes(
            T, H, E, I, Is, case["k"], has_shared=Is > 0,
            wdtype=1 if kind == "bf16" else 0))
    state["out"] = _result(case)
    return state


def run(state):
    case, x, out = state["case"], state["x"], state["out"]
    kind, T = case["kind"], case["T"]
    if kind == "fp8":
        _fp8.fp8_gemm_dev(x, state["w"], state["s"], out, T, case["N"], case["K"])
    elif kind == "fp4":
        _ds.fp4_moe_linear_dev(x, state["w"], state["s"], out, T, case["N"], case["K"])
    elif kind == "dense":
        state["mlp"].forward_dev(x, out, T)
    elif kind == "ds":
        _moe.deepseek_forward_dev(
            x, out, state["w"], **_sizes(case), out_f32=_decode(case),
            n_group=N_GROUP, topk_group=TOPK_GROUP, scoring="sigmoid",
            route_scale=ROUTE_SCALE, swiglu_limit=LIMIT, workspace=state["ws"])
    elif "stack" in state:
        state["stack"].moe_dev(x, out, 0, T)
    else:
        _moe.qwen_forward_dev(x, out, state["w"], **_sizes(case),
                              out_f32=_decode(case),
                              wdtype=1 if kind == "bf16" else 0,
                              workspace=state["ws"])
    return out


# ---------------------------------------------------------------------------
# the same values in 64 bits
# ---------------------------------------------------------------------------

def _fp8_exact(q, s):
    w = q.view(torch.float8_e4m3fn).double()
    s = s.double().repeat_interleave(128, 0)[:w.shape[0]]
    return w * s.repeat_interleave(128, 1)[:, :w.shape[1]]


def _fp4_exact(p, s):
    value = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device=GPU)
    value = torch.cat([value, -value])
    w = torch.stack([value[(p & 15).int()], value[(p >> 4).int()]], -1)
    w = w.view(p.shape[0], -1, 32) * torch.exp2(s.double() - 127)[..., None]
    return w.view(p.shape[0], -1)


def _quantized(x, pow2):
    """x through e4m3 with a scale for each row and 128 columns. The scale
    and the quotient are fp32 values by the format's definition (a tie of the
    rounding is decided there); what comes back is exact."""
    b = x.float().view(x.shape[0], -1, 128)
    s = b.abs().amax(-1, keepdim=True).clamp_min(1e-4) * (1.0 / 448.0)
    if pow2:
        s = torch.exp2(torch.ceil(torch.log2(s.double()))).float()
    q = (b / s).clamp(-448, 448).to(torch.float8_e4m3fn).double()
    return (q * s.double()).view(x.shape)


def _expert_exact(x, wg, wu, wd, weight, limit, quant, pow2, late):
    """One SwiGLU expert's weighted rows; prompts quantize the rows that meet
    FP8 and MXFP4 weights, the weight applied before (DeepSeek) or after."""
    gate, up = x @ wg.T, x @ wu.T
    if limit:
        up, gate = up.clamp(-limit, limit), gate.clamp(max=limit)
    h = gate * torch.sigmoid(gate) * up
    if not late:
        h = h * weight
    y = (_quantized(h, pow2) if quant else h) @ wd.T
    return y * weight if late else y


def _routed_exact(out, x, ids, weight, expert, **how):
    for e in torch.unique(ids).tolist():
        t, j = torch.nonzero(ids == e, as_tuple=True)
        out.index_add_(0, t, _expert_exact(x[t], *expert(e), weight[t, j][:, None], **how))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("fp8", "fp4"):
        w, s, x = _linear_inputs(case, seed)
        w = _fp8_exact(w, s) if kind == "fp8" else _fp4_exact(w, s)
        return x.double() @ w.T
    quant = not _decode(case)
    if kind == "dense":
        w, x = _dense_inputs(case, seed)
        wg, wu, wd = (_fp8_exact(w[n], w[n + "_s"]) for n in ("wg", "wu", "wd"))
        return _expert_exact(x.double(), wg, wu, wd, 1.0, 0.0, False, False, True)
    T, H, E, I, k = case["T"], case["H"], case["E"], case["I"], case["k"]
    w, x = (_ds_inputs if kind == "ds" else _qwen_inputs)(case, seed)
    x = x.double()
    logits = x @ w["router_w"].double().T
    pow2 = kind == "ds"
    xe = _quantized(x, pow2) if quant else x
    out = torch.zeros(T, H, dtype=torch.float64, device=GPU)
    how = {"quant": quant, "pow2": pow2}
    if kind == "ds":
        score = torch.sigmoid(logits)
        biased = score + w["bias"].double()
        group = biased.view(T, N_GROUP, -1).topk(2, -1).values.sum(-1)
        keep = torch.zeros_like(group, dtype=torch.bool)
        keep.scatter_(1, group.topk(TOPK_GROUP, -1).indices, True)
        biased = biased.masked_fill(~keep.repeat_interleave(E // N_GROUP, 1), -1e30)
        ids = biased.topk(k, -1).indices
        weight = score.gather(1, ids)
        weight = weight / weight.sum(-1, keepdim=True) * ROUTE_SCALE

        def expert(e):
            return [_fp4_exact(w[n][e * r:(e + 1) * r], w[n + "_s"][e * r:(e + 1) * r])
                    for n, r in (("w1", I), ("w3", I), ("w2", H))]
        # decode scales the expert's result, prompts its quantized hidden row
        _routed_exact(out, xe, ids, weight, expert, limit=LIMIT, late=not quant, **how)
        shared = [_fp8_exact(w[n], w[n + "_s"]) for n in ("s1", "s3", "s2")]
        out += _expert_exact(xe, *shared, 1.0, LIMIT, late=True, **how)
        return out
    if "router_bias" in w:
        logits = logits + w["router_bias"].double()
    p = torch.softmax(logits, -1)
    weight, ids = p.topk(k, -1)
    weight = weight / (weight.sum(-1, keepdim=True) + 1e-20)

    def rows(name, e, r):
        if kind == "bf16":
            return w[name][e].double()
        b = r // 128
        return _fp8_exact(w[name][e * r:(e + 1) * r], w[name + "_s"][e * b:(e + 1) * b])

    def expert(e):
        return rows("wg", e, I), rows("wu", e, I), rows("wd", e, H)
    _routed_exact(out, xe, ids, weight, expert, limit=0.0, late=True, **how)
    if case["Is"]:
        if kind == "bf16":
            shared = [w[n].double() for n in ("sg", "su", "sd")]
        else:
            shared = [_fp8_exact(w[n], w[n + "_s"]) for n in ("sg", "su", "sd")]
        gate = torch.sigmoid(x @ w["sgl"].double())[:, None]
        out += _expert_exact(xe, *shared, gate, 0.0, late=True, **how)
    return out


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------

def work(case):
    """Each weight of a touched expert (those a uniform routing of T * k
    assignments touches), of the shared expert and of the router once, the
    activations once, the result once."""
    kind, T = case["kind"], case["T"]
    if kind in ("fp8", "fp4"):
        N, K = case["N"], case["K"]
        per = 1.0 if kind == "fp8" else 0.5 + 1 / 32
        return {"bytes": N * K * per + 4 * T * (N + K), "flops": 2.0 * T * N * K}
    H, I = case["H"], case["I"]
    result = (4 if _decode(case) else 2) * T * H
    if kind == "dense":
        return {"bytes": 3.0 * H * I + 2 * T * H + result, "flops": 6.0 * T * H * I}
    E, Is, k = case["E"], case["Is"], case["k"]
    per = {"qwen": 1.0, "ds": 0.5 + 1 / 32, "bf16": 2.0}[kind]
    shared = {"qwen": 1.0, "ds": 1.0, "bf16": 2.0}[kind]
    touched = E * (1.0 - (1.0 - 1.0 / E) ** (T * k))
    if case.get("skew"):
        touched = min(touched, E - E // 20)
    return {"bytes": 3 * H * (touched * I * per + Is * shared) + 2 * E * H + 2 * T * H + result,
            "flops": 6.0 * T * H * (k * I + Is) + 2.0 * T * H * E}


def tolerance(case):
    """About four times what the path is off `exact` (prompts 2.5e-3 to
    2.8e-3: e4m3 rows, a bf16 row for each assignment and a bf16 result;
    decode 2.4e-6: sums in fp32, the hidden row in two bf16 parts), and what
    another order of their fp32 sums gives the bf16 layer and the linears
    (2e-7 to 1.4e-6 off `exact`). "max" leaves room for one near tie of the
    routing or of the e4m3 rounding."""
    if not _decode(case) and case["kind"] in ("qwen", "ds"):
        return {"rel": 1e-2, "max": 0.5}
    return {"rel": 1e-5, "max": 4e-4}
