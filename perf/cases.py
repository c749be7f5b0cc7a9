"""Timed cases of the mixture-of-experts layers: what a serving program has them do.

A case names a layer shape, an entry point and a token count:

  entry "layer"     the layer module (FP8BlockMoE, or MXFP4MoE for "gpt_oss"), decode or
                    prefill, with or without the layer's own RMSNorm and residual add
  entry "block_tkg" the decode operator moe_block_tkg (norm, router and experts in one call)
  entry "cte"       the prefill operators in a row: router, build_blockwise_mapping, moe_cte

Inputs are synthetic: activations N(0, 1) in bf16, router weight N(0, 0.02), expert weights
N(0, 0.02) quantized to the checkpoint formats (e4m3fn with 128x128 fp32 scales, or MXFP4
with one E8M0 byte per 32 values), gamma 1 + N(0, 0.1), biases N(0, 0.1), and with "zipf" a
Zipf(1.2) bias on the router logits that leaves a tenth of the experts nearly without tokens.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "vllm-neuron_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

FP8 = torch.float8_e4m3fn
DEV = "cuda"

# hidden, expert intermediate, experts, top-k, shared experts, groups, kept groups, scale
_FP8_SHAPES = {
    "small": dict(H=1024, I=512, E=8, K=2, S=0),
    "dsv3": dict(H=7168, I=2048, E=256, K=8, S=1, groups=8, kept=4, scale=2.5),
    "kimi_k2": dict(H=7168, I=2048, E=384, K=8, S=1, groups=1, kept=1, scale=2.827),
    "glm45": dict(H=5120, I=1536, E=160, K=8, S=1, groups=1, kept=1, scale=2.5),
}
# hidden and intermediate padded to a multiple of 256 from h_real / i_real
_MX_SHAPES = {"gpt_oss": dict(H=3072, I=3072, E=128, K=4, S=0, h_real=2880, i_real=2880)}


def _shape(case):
    return {**_FP8_SHAPES, **_MX_SHAPES}[case["model"]]


def _is_mx(case):
    return case["model"] in _MX_SHAPES


def _case(name, model, tokens, entry="layer", norm=True, residual=False, decode=True, zipf=False):
    return dict(name=name, model=model, entry=entry, tokens=tokens, norm=norm, residual=residual,
                decode=decode, zipf=zipf)


def listed():
    return [
        # the smallest layer, a full decode batch: all launches and host work
        _case("small_decode_64", "small", 64, norm=False),
        # one user's decode step: 9 of 385 experts, latency and their weight stream
        _case("kimi_k2_decode_1", "kimi_k2", 1),
        _case("gpt_oss_decode_1", "gpt_oss", 1),
        # decode batches: nearly every expert is read for a few rows
        _case("dsv3_decode_64", "dsv3", 64),
        _case("gpt_oss_decode_61", "gpt_oss", 61),
        # the decode operator on a ragged batch
        _case("glm45_block_tkg_13", "glm45", 13, entry="block_tkg"),
        # a short prompt: tens of rows per expert
        _case("kimi_k2_prefill_2048", "kimi_k2", 2048, residual=True, decode=False),
        _case("gpt_oss_prefill_2048", "gpt_oss", 2048, residual=True, decode=False),
        # the prefill operators on a ragged prompt
        _case("glm45_cte_1500", "glm45", 1500, entry="cte", norm=False, decode=False),
        # a prompt with skewed routing: experts of thousands of rows next to empty ones
        _case("glm45_zipf_prefill_4001", "glm45", 4001, norm=False, decode=False, zipf=True),
        # full prefill chunks: hundreds of rows per expert
        _case("gpt_oss_prefill_8192", "gpt_oss", 8192, residual=True, decode=False),
        _case("dsv3_prefill_8192", "dsv3", 8192, residual=True, decode=False),
    ]


def draw(rng):
    model, lo, hi = rng.choice([("small", 1, 8192), ("dsv3", 1, 7000), ("kimi_k2", 1, 4500),
                                ("glm45", 1, 8192), ("gpt_oss", 1, 8192), ("gpt_oss", 1, 8192)])
    tokens = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if tokens > 16 and rng.random() < 0.7:
        tokens |= 1
    entry = "layer"
    if model != "gpt_oss" and rng.random() < 0.3:
        entry = "block_tkg" if tokens <= 256 else "cte"
    decode = tokens <= 256
    norm = entry == "block_tkg" or (entry == "layer" and rng.random() < 0.7)
    residual = norm and not decode and entry == "layer" and rng.random() < 0.6
    zipf = entry == "layer" and model in ("glm45", "kimi_k2") and rng.random() < 0.4
    return dict(model=model, entry=entry, tokens=tokens, norm=norm, residual=residual,
                decode=decode, zipf=zipf)


# ------------------------------------------------------------------ inputs (plain torch)

def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * std


def _quant_128x128(w):
    O, K = w.shape
    b = w.view(O // 128, 128, K // 128, 128)
    s = b.abs().amax(dim=(1, 3)) / 448.0
    q = (b / s[:, None, :, None]).clamp_(-448.0, 448.0).to(FP8)
    return q.view(O, K), s


_FP4_MIDS = (0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0)
_FP4_LEVELS = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _mx_exp(amax, emax):
    """floor(log2(amax)) - emax, at least -127."""
    return torch.clamp((torch.frexp(amax)[1] - 1 - emax), min=-127)


def _quant_mxfp4(w):
    O, K = w.shape
    b = w.view(O, K // 32, 32)
    amax = b.abs().amax(-1)
    e = torch.where(amax > 0, _mx_exp(amax, 2), torch.full_like(amax, -127, dtype=torch.int32))
    v = b * torch.exp2(-e.float()).unsqueeze(-1)
    mids = torch.tensor(_FP4_MIDS, device=DEV)
    code = torch.bucketize(v.abs(), mids, out_int32=True).to(torch.uint8)
    code |= (v < 0).to(torch.uint8) << 3
    code = code.view(O, K)
    return code[:, 0::2] | (code[:, 1::2] << 4), (e + 127).to(torch.uint8)


def _fp8_weights(d, g, n):
    H, I = d["H"], d["I"]
    out = (torch.empty(n, 2 * I, H, dtype=FP8, device=DEV),
           torch.empty(n, 2 * I // 128, H // 128, device=DEV),
           torch.empty(n, H, I, dtype=FP8, device=DEV),
           torch.empty(n, H // 128, I // 128, device=DEV))
    for e in range(n):
        out[0][e], out[1][e] = _quant_128x128(_randn(g, 2 * I, H, std=0.02))
        out[2][e], out[3][e] = _quant_128x128(_randn(g, H, I, std=0.02))
    return out


def _mx_weights(d, g):
    H, I, E, hr, ir = d["H"], d["I"], d["E"], d["h_real"], d["i_real"]
    w13 = torch.empty(E, 2 * I, H // 2, dtype=torch.uint8, device=DEV)
    s13 = torch.empty(E, 2 * I, H // 32, dtype=torch.uint8, device=DEV)
    w2 = torch.empty(E, H, I // 2, dtype=torch.uint8, device=DEV)
    s2 = torch.empty(E, H, I // 32, dtype=torch.uint8, device=DEV)
    for e in range(E):
        a = _randn(g, 2, I, H, std=0.02)
        a[:, ir:], a[:, :, hr:] = 0, 0
        b = _randn(g, H, I, std=0.02)
        b[hr:], b[:, ir:] = 0, 0
        w13[e], s13[e] = _quant_mxfp4(a.view(2 * I, H))
        w2[e], s2[e] = _quant_mxfp4(b)
    b13 = _randn(g, E, 2, I, std=0.1)
    b13[:, 1] += 1.0
    b13[:, :, ir:] = 0
    b2 = _randn(g, E, H, std=0.1)
    b2[:, hr:] = 0
    return w13, s13, b13.view(E, 2 * I), w2, s2, b2


def _inputs(case, seed):
    d = _shape(case)
    H, E, T = d["H"], d["E"], case["tokens"]
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    hr = d.get("h_real", H)
    t = {"x": _randn(g, T, H).to(torch.bfloat16), "router": _randn(g, E, H, std=0.02).to(torch.bfloat16)}
    t["x"][:, hr:] = 0
    t["router"][:, hr:] = 0
    if case["norm"]:
        t["gamma"] = 1.0 + _randn(g, H, std=0.1)
    if case["residual"]:
        t["residual"] = _randn(g, T, H).to(torch.bfloat16)
        t["residual"][:, hr:] = 0
    if _is_mx(case):
        t["router_bias"] = _randn(g, E, std=0.1)
        t["experts"] = _mx_weights(d, g)
        return t
    if "groups" in d:
        t["corr"] = _randn(g, E, std=0.01)
    if case["zipf"]:
        p = torch.arange(1, E + 1, device=DEV, dtype=torch.float64) ** -1.2
        bias = torch.log(p / p.sum())
        bias[E - E // 10:] = -1e4
        t["router_bias"] = bias.float()[torch.randperm(E, generator=g, device=DEV)]
    t["experts"] = _fp8_weights(d, g, E)
    if d["S"] and case["entry"] == "layer":
        t["shared"] = _fp8_weights(d, g, d["S"])
    return t


# ------------------------------------------------------------------ the calls

def prepare(case, seed):
    from vllm_neuron_amd import PRESETS
    from vllm_neuron_amd.layer import FP8BlockMoE
    from vllm_neuron_amd.layer_mx import MXFP4MoE
    from vllm_neuron_amd.weights import Fp8MoEWeights
    from vllm_neuron_amd.weights_mx import MxMoEWeights

    t = _inputs(case, seed)
    d = _shape(case)
    state = {"case": case, "x": t["x"], "residual": t.get("residual")}
    if case["entry"] == "layer" and _is_mx(case):
        w13, s13, b13, w2, s2, b2 = t["experts"]
        w = MxMoEWeights(router_w=t["router"], w13=w13, w13_scale=s13, b13=b13, w2=w2,
                         w2_scale=s2, b2=b2, router_bias=t["router_bias"])
        state["layer"] = MXFP4MoE(w, d["K"], norm_weight=t.get("gamma"), eps=1e-5,
                                  hidden_actual=d["h_real"] if case["norm"] else None)
    elif case["entry"] == "layer":
        w13, s13, w2, s2 = t["experts"]
        kw = {}
        if "shared" in t:
            kw = dict(zip(("shared_w13", "shared_w13_scale", "shared_w2", "shared_w2_scale"),
                          t["shared"]))
        w = Fp8MoEWeights(router_w=t["router"], w13=w13, w13_scale=s13, w2=w2, w2_scale=s2,
                          router_bias=t.get("router_bias"), corr_bias=t.get("corr"), **kw)
        state["layer"] = FP8BlockMoE(PRESETS[case["model"]], w, norm_weight=t.get("gamma"))
    else:
        # the stacked checkpoint layout, which the operators take as it is
        state["experts"] = t["experts"]
        state["router_t"] = t["router"].t()
        state["gamma"] = t.get("gamma")
        state["top_k"] = d["K"]
    return state


def run(state):
    from vllm_neuron_amd.functional import moe as M

    case, x = state["case"], state["x"]
    if case["entry"] == "layer":
        return state["layer"](x, is_decode=case["decode"], residual=state["residual"])
    w13, s13, w2, s2 = state["experts"]
    if case["entry"] == "block_tkg":
        return M.moe_block_tkg(
            x, state["gamma"], state["router_t"], w13, w2, top_k=state["top_k"],
            expert_gate_up_weights_scale=s13, expert_down_weights_scale=s2,
            router_act_fn=M.RouterActFnType.SIGMOID, norm_topk_prob=True,
            expert_affinities_scaling_mode=M.ExpertAffinityScaleMode.POST_SCALE)
    E, K = w13.shape[0], state["top_k"]
    affinities = M.router(x, state["router_t"], K)
    masked, tpid, b2e, _ = M.build_blockwise_mapping(affinities, E, K, 256)
    out = M.moe_cte(x, masked, w13, w2, tpid, b2e, 256, M.MoECTEImplementation.shard_on_block,
                    gate_up_proj_scale=s13, down_proj_scale=s2)
    return out, affinities


def work(case):
    """Bytes: the experts that T tokens reach (at even routing), the router weight, each
    input row read and each output row written once. Flops: the router product and three
    H x I products per (token, expert) pair."""
    d, T = _shape(case), case["tokens"]
    H, I, E, K = d["H"], d["I"], d["E"], d["K"]
    S = d["S"] if case["entry"] == "layer" else 0
    active = E * (1.0 - (1.0 - K / E) ** T) + S
    if _is_mx(case):
        per_expert = 3 * H * I * (0.5 + 1 / 32) + 4 * (2 * I + H)
    else:
        per_expert = 3 * H * I * (1 + 4 / 16384)
    rows = T * H * 2 * (4 if case["residual"] else 2)
    if case["entry"] != "layer":
        rows += 4 * T * E  # the router's fp32 logits or affinities are an output
    return {"bytes": active * per_expert + 2 * E * H + rows,
            "flops": 2.0 * T * H * E + 6.0 * T * (K + S) * H * I}


def tolerance(case):
    # bf16 outputs of 8-bit operands. Against exact() the paths sit 2.3e-3 to 2.8e-3 away
    # (the roundings of y and out to bf16, and activation codes that round the other way), up to
    # 5.6e-3 at 8192 tokens, where a token's near-tie between two experts may go the other way.
    return {"rel": 1e-2}


# ------------------------------------------------------------------ float64 restatement

def _e4m3(v):
    return v.clamp(-448.0, 448.0).float().to(FP8).double()


def _act_1x128(v):
    """v rounded to e4m3 codes with one scale per 128 columns. The scale and the quotient
    are fp32 by the format's definition: bf16 inputs meet exact ties between two codes,
    which any other rounding of the quotient would break differently."""
    R, C = v.shape
    b = v.float().view(R, C // 128, 128)
    amax = b.abs().amax(-1, keepdim=True).clamp(min=1e-10)
    s = amax / torch.full_like(amax, 448.0)
    return (_e4m3(b / s) * s.double()).view(R, C)


def _act_mx(v):
    R, C = v.shape
    b = v.view(R, C // 32, 32)
    amax = b.abs().amax(-1, keepdim=True)
    e = torch.where(amax > 0, _mx_exp(amax, 8), torch.full_like(amax, -127).int()).double()
    return (_e4m3(b * torch.exp2(-e)) * torch.exp2(e)).view(R, C)


def _deq_fp8(q, s):
    O, K = q.shape
    return (q.double().view(O // 128, 128, K // 128, 128)
            * s.double()[:, None, :, None]).view(O, K)


def _deq_fp4(q, s):
    O, half = q.shape
    code = torch.stack((q & 15, q >> 4), dim=-1).view(O, 2 * half).long()
    lv = torch.tensor(_FP4_LEVELS, device=DEV, dtype=torch.float64)
    v = lv[code & 7] * torch.where(code >= 8, -1.0, 1.0).double()
    scale = torch.exp2(s.double() - 127.0)
    return (v.view(O, half // 16, 32) * scale[..., None]).view(O, 2 * half)


def _route(case, d, logits, corr):
    """(ids, weights) of each token's experts."""
    T, E, K = logits.shape[0], d["E"], d["K"]
    if case["entry"] == "block_tkg":
        act = torch.sigmoid(logits)
        w, ids = act.topk(K, dim=-1)
        return ids, w / (w.sum(-1, keepdim=True) + 1e-20)
    if "groups" not in d or case["entry"] == "cte":
        v, ids = logits.topk(K, dim=-1)
        return ids, torch.softmax(v, -1)
    act = torch.sigmoid(logits)
    key = act + corr.double()
    if d["groups"] > 1:
        grp = key.view(T, d["groups"], -1)
        keep = grp.topk(2, dim=-1)[0].sum(-1).topk(d["kept"], dim=-1)[1]
        mask = torch.zeros(T, d["groups"], device=DEV, dtype=torch.bool).scatter_(1, keep, True)
        key = grp.masked_fill(~mask[..., None], -math.inf).view(T, E)
    ids = key.topk(K, dim=-1)[1]
    w = act.gather(1, ids)
    return ids, w / (w.sum(-1, keepdim=True) + 1e-20) * d["scale"]


def exact(case, seed):
    t, d = _inputs(case, seed), _shape(case)
    H, I, E = d["H"], d["I"], d["E"]
    x, res_out = t["x"].double(), None
    if case["residual"]:
        x = (x + t["residual"].double()).to(torch.bfloat16).double()
        res_out = x
    if case["norm"]:
        n = d.get("h_real", H)
        rn = torch.rsqrt(x[:, :n].square().mean(-1, keepdim=True)
                         + (1e-5 if _is_mx(case) else 1e-6))
        x = x * rn * t["gamma"].double()
        x[:, n:] = 0
        x = x.to(torch.bfloat16).double()
    logits = x @ t["router"].double().t()
    if "router_bias" in t:
        logits += t["router_bias"].double()
    ids, wts = _route(case, d, logits, t.get("corr"))
    mx = _is_mx(case)
    act = _act_mx if mx else _act_1x128
    xq = act(x)
    out = torch.zeros_like(x)

    def add(e, weights, rows, scale):
        if mx:
            w13, s13, b13, w2, s2, b2 = weights
            gu = xq[rows] @ _deq_fp4(w13[e], s13[e]).t() + b13[e].double()
            gate, up = gu[:, :I].clamp(max=7.0), gu[:, I:].clamp(-6.0, 8.0)
            h = gate * torch.sigmoid(1.702 * gate) * up
            y = act(h) @ _deq_fp4(w2[e], s2[e]).t() + b2[e].double()
        else:
            w13, s13, w2, s2 = weights
            gu = xq[rows] @ _deq_fp8(w13[e], s13[e]).t()
            gate, up = gu[:, :I], gu[:, I:]
            y = act(gate * torch.sigmoid(gate) * up) @ _deq_fp8(w2[e], s2[e]).t()
        out.index_add_(0, rows, y * scale[:, None])

    for e in range(E):
        rows, k = (ids == e).nonzero(as_tuple=True)
        if rows.numel():
            add(e, t["experts"], rows, wts[rows, k])
    if "shared" in t:
        rows = torch.arange(x.shape[0], device=DEV)
        for j in range(d["S"]):
            add(j, t["shared"], rows, torch.ones(x.shape[0], device=DEV, dtype=torch.float64))
    if case["entry"] == "block_tkg":
        return out, logits
    if case["entry"] == "cte":
        return out, torch.zeros_like(logits).scatter_(1, ids, wts)
    return out if res_out is None else (out, res_out)
