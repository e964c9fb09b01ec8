"""Workloads whose speed is watched: what a user of the framework has it do, through its public entry points, at the
sizes of the Llama-3-8B, Qwen2.5-7B and Mixtral-8x7B layers that the tests and the benchmark use.

    listed()            twelve fixed cases, smallest call to largest layer
    draw(rng)           one more case out of the same ranges
    prepare(case, seed) weights, inputs, caches: what a program holds before the call
    run(state)          one pass
    work(case)          bytes and flops a pass cannot do without
    tolerance(case)     how far another correct implementation's results may lie

Kinds of cases:
    norm     agemm.rmsnorm_quantize_x: the fused RMSNorm -> FP4 quantizer in front of every projection
    linear   one ARC linear from bf16 to bf16: layers.quantize_tokens, then layers.QLinearLayer
    prefill  a Llama decoder layer on whole prompts (fused qkv and gate_up projections, fused norms)
    qwen     a Qwen2 decoder layer built from its own linears and calibration entries, as a converted checkpoint is:
             separate projections, q / k / v bias, the model's norms in front of the quantizers
    decode   one token per sequence through a Llama decoder layer over the INT4 paged KV cache, launched from Python
             or replayed as a captured graph
    moe      a Mixtral feed-forward block: routing, grouped expert MLPs, combination
"""
import math

import torch
import torch.nn as nn

from arcquant_amd import agemm, layers
from arcquant_amd.kv_cache import MultiLayerPagedKVCache4Bit

EPS = 1e-5
HIDDEN, INTER, HEADS, KV_HEADS, HEAD_DIM = 4096, 14336, 32, 8, 128                  # Llama-3-8B
Q_HIDDEN, Q_INTER, Q_HEADS, Q_KV_HEADS = 3584, 18944, 28, 4                         # Qwen2.5-7B
EXPERTS, TOP_K = 8, 2                                                               # Mixtral-8x7B
PROJECTIONS = [(6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336)]            # qkv, o, gate_up, down: N x K
GROUP = {"NVFP4": 16, "MXFP4": 32}


def listed():
    return [
        # the smallest call there is: one token's norm while a single sequence is generated
        {"name": "norm_token", "kind": "norm", "fmt": "NVFP4", "rows": 1, "k": 4096, "select": 64},
        # the same operator on a prompt batch: the quantizer at memory speed
        {"name": "norm_prompt", "kind": "norm", "fmt": "NVFP4", "rows": 4096, "k": 4096, "select": 256},
        # a linear of a small decode batch: a stream of its weights (gate_up)
        {"name": "linear_decode", "kind": "linear", "fmt": "NVFP4", "rows": 16, "n": 28672, "k": 4096, "select": 256},
        # a few short prompts, odd token count: neither a weight stream nor large tiles (qkv)
        {"name": "linear_short", "kind": "linear", "fmt": "NVFP4", "rows": 333, "n": 6144, "k": 4096, "select": 128},
        # a large linear in the format the matrix cores scale by themselves (down)
        {"name": "linear_large", "kind": "linear", "fmt": "MXFP4", "rows": 4096, "n": 4096, "k": 14336, "select": 256},
        # prompts through a layer: the largest case of either format
        {"name": "prefill_nv", "kind": "prefill", "fmt": "NVFP4", "batch": 8, "seq": 2048},
        {"name": "prefill_mx", "kind": "prefill", "fmt": "MXFP4", "batch": 4, "seq": 1024},
        # a converted checkpoint's layer on ragged prompts
        {"name": "qwen_prompt", "kind": "qwen", "fmt": "NVFP4", "batch": 3, "seq": 777},
        # serving: one token of 64 sequences, the step captured once and replayed
        {"name": "decode_graph", "kind": "decode", "fmt": "NVFP4", "batch": 64, "kv": 2048, "graph": True},
        # interactive generation from Python: few sequences, launches and host work count
        {"name": "decode_eager", "kind": "decode", "fmt": "MXFP4", "batch": 8, "kv": 1000, "graph": False},
        # mixture of experts: a prompt batch, and a decode batch (few rows per expert, every expert's weights read)
        {"name": "moe_prompt", "kind": "moe", "fmt": "NVFP4", "tokens": 4096},
        {"name": "moe_decode", "kind": "moe", "fmt": "NVFP4", "tokens": 64},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["norm", "linear", "linear", "prefill", "qwen", "decode", "decode", "moe"])
    fmt = rng.choice(["NVFP4", "MXFP4"])
    if kind == "norm":
        return {"kind": kind, "fmt": fmt, "rows": _log_int(rng, 1, 16384), "k": rng.choice([2048, 3072, 4096]),
                "select": rng.choice([64, 128, 256])}
    if kind == "linear":
        n, k = rng.choice(PROJECTIONS)
        return {"kind": kind, "fmt": fmt, "rows": _log_int(rng, 1, 4096), "n": n, "k": k,
                "select": rng.choice([128, 256])}
    if kind == "prefill":
        return {"kind": kind, "fmt": fmt, "batch": rng.randint(1, 8), "seq": _log_int(rng, 100, 2048)}
    if kind == "qwen":
        return {"kind": kind, "fmt": fmt, "batch": rng.randint(1, 4), "seq": _log_int(rng, 100, 2048)}
    if kind == "decode":
        return {"kind": kind, "fmt": fmt, "batch": _log_int(rng, 1, 64), "kv": _log_int(rng, 100, 4000),
                "graph": rng.random() < 0.5}
    return {"kind": kind, "fmt": fmt, "tokens": _log_int(rng, 1, 4096)}


# ------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _activations(rows, k, g, outliers=0.01, gain=40.0):
    """~N(0,1) with a small share of outlier channels, bf16"""
    x = torch.randn(rows, k, generator=g, device="cuda")
    cols = torch.randperm(k, generator=g, device="cuda")[:max(1, round(outliers * k))]
    x[:, cols] *= gain
    return x.to(torch.bfloat16)


def _order(x):
    """calibrated channel order: ascending per-channel maxima (outliers last)"""
    return torch.argsort(x.float().abs().amax(0), stable=True).to(torch.int16)


def _any_order(k, g):
    return torch.randperm(k, generator=g, device="cuda").to(torch.int16)


def _gamma(k, g):
    return (torch.rand(k, generator=g, device="cuda") + 0.5).to(torch.bfloat16)


def _linear(n, k, g, bias=False):
    lin = nn.Linear(k, n, bias=bias, device="meta", dtype=torch.bfloat16)
    lin.weight = nn.Parameter((torch.randn(n, k, generator=g, device="cuda") * 0.02).to(torch.bfloat16), requires_grad=False)
    if bias:
        lin.bias = nn.Parameter((torch.randn(n, generator=g, device="cuda") * 0.1).to(torch.bfloat16), requires_grad=False)
    return lin


def _normed(x, gamma):
    h = x.float()
    return (h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + EPS)).to(torch.bfloat16) * gamma


class _LlamaLayer:
    """layers.LlamaDecoderLayer assembled from weights that are on the GPU already"""

    def __init__(self, x, fmt, g, select=256):
        g1, g2 = _gamma(HIDDEN, g), _gamma(HIDDEN, g)
        attn_in, mlp_in = _order(_normed(x, g1)), _order(_normed(x, g2))
        self.input_layernorm = layers.RMSNormQuant(g1, EPS, select, attn_in, fmt)
        self.post_attention_layernorm = layers.RMSNormQuant(g2, EPS, select, mlp_in, fmt)
        self.self_attn = layers.LlamaAttention(_linear((HEADS + 2 * KV_HEADS) * HEAD_DIM, HIDDEN, g), _linear(HIDDEN, HIDDEN, g),
                                               HEADS, KV_HEADS, select, select, attn_in, _any_order(HIDDEN, g), fmt)
        self.mlp = layers.LlamaMLP(_linear(2 * INTER, HIDDEN, g), _linear(HIDDEN, INTER, g), select, select, mlp_in,
                                   _any_order(INTER, g), fmt)

    def __call__(self, x, kv_cache=None, past_len=0, layer_idx=0):
        h = self.self_attn(self.input_layernorm(x), kv_cache, past_len, layer_idx, residual=x)
        return self.mlp(self.post_attention_layernorm(h), residual=h)


def prepare(case, seed):
    kind, fmt, g = case["kind"], case["fmt"], _gen(seed)
    s = {"kind": kind, "fmt": fmt}
    if kind == "norm":
        k = case["k"]
        x = _activations(case["rows"], k, g, 0.005, 50.0)
        gamma = _gamma(k, g)
        s.update(x=x, gamma=gamma, order=_order(_normed(_activations(256, k, g, 0.005, 50.0), gamma)), select=case["select"])
    elif kind == "linear":
        x = _activations(case["rows"], case["k"], g)
        order = _order(x)
        s.update(x=x, order=order, select=case["select"],
                 linear=layers.QLinearLayer(_linear(case["n"], case["k"], g), case["select"], order, quant_type=fmt))
    elif kind == "prefill":
        x = _activations(case["batch"] * case["seq"], HIDDEN, g)
        s.update(x=x.view(case["batch"], case["seq"], HIDDEN), layer=_LlamaLayer(x[:2048], fmt, g))
    elif kind == "qwen":
        x = _activations(case["batch"] * case["seq"], Q_HIDDEN, g)
        norms = [_gamma(Q_HIDDEN, g), _gamma(Q_HIDDEN, g)]
        kv = Q_KV_HEADS * HEAD_DIM
        lin = {"q_proj": _linear(Q_HIDDEN, Q_HIDDEN, g, True), "k_proj": _linear(kv, Q_HIDDEN, g, True),
               "v_proj": _linear(kv, Q_HIDDEN, g, True), "o_proj": _linear(Q_HIDDEN, Q_HIDDEN, g),
               "gate_proj": _linear(Q_INTER, Q_HIDDEN, g), "up_proj": _linear(Q_INTER, Q_HIDDEN, g),
               "down_proj": _linear(Q_HIDDEN, Q_INTER, g)}
        attn_in, mlp_in = _order(_normed(x[:2048], norms[0])), _order(_normed(x[:2048], norms[1]))
        order = {"self_attn.q_proj": attn_in, "self_attn.k_proj": attn_in, "self_attn.v_proj": attn_in,
                 "self_attn.o_proj": _any_order(Q_HIDDEN, g), "mlp.gate_proj": mlp_in, "mlp.up_proj": mlp_in,
                 "mlp.down_proj": _any_order(Q_INTER, g)}
        order = {f"layers.0.{name}.input": v for name, v in order.items()}
        select = {name: 128 for name in order}
        s.update(x=x.view(case["batch"], case["seq"], Q_HIDDEN),
                 layer=layers.QQwen2DecoderLayer(lin, norms, EPS, Q_HEADS, Q_KV_HEADS, select, order, 0, fmt))
    elif kind == "decode":
        batch, kv = case["batch"], case["kv"]
        x = _activations(batch, HIDDEN, g)
        layer = _LlamaLayer(_activations(256, HIDDEN, g), fmt, g)
        # sequences of kv - 1 cached tokens; the step's token takes slot kv (the same one in every pass, as in the
        # second and later layers of a model, which run on a cache that the first one has advanced)
        cache = MultiLayerPagedKVCache4Bit(batch, 16, kv + 16, "cuda", 1, KV_HEADS, HEAD_DIM, dtype=torch.bfloat16)
        k, v = (torch.randn(batch, kv - 1, KV_HEADS, HEAD_DIM, generator=g, device="cuda").to(torch.bfloat16) for _ in "kv")
        cache.update(k, v, 0)
        del k, v
        cache.external_step = True
        s.update(x=x.view(batch, 1, HIDDEN), layer=layer, cache=cache, step=None)
        if case["graph"]:
            s["step"] = layers.GraphedDecodeStep(layer, cache, batch, HIDDEN, advance=False)
            s["step"].x.copy_(s["x"])          # where the previous layer's output would be
        cache.begin_step()
    elif kind == "moe":
        tokens, select = case["tokens"], 128
        x = _activations(tokens, HIDDEN, g)
        skew = torch.log(1.0 / torch.arange(1, EXPERTS + 1, device="cuda").float() ** 1.1)      # Zipf over the experts
        logits = torch.randn(tokens, EXPERTS, generator=g, device="cuda") + skew
        experts = []
        for _ in range(EXPERTS):
            order = _order(_activations(256, HIDDEN, g))
            experts.append(layers.MixtralExpertMLP(_linear(INTER, HIDDEN, g), _linear(INTER, HIDDEN, g),
                                                   _linear(HIDDEN, INTER, g), select, order, _any_order(INTER, g), fmt))
        s.update(x=x.view(1, tokens, HIDDEN), logits=logits,
                 block=layers.MixtralSparseMoeBlock(_linear(EXPERTS, HIDDEN, g), experts, TOP_K))
    else:
        raise ValueError(f"unknown kind {kind!r}")
    return s


@torch.no_grad()
def run(s):
    kind = s["kind"]
    if kind == "norm":
        return agemm.rmsnorm_quantize_x(s["x"], s["gamma"], EPS, s["order"], s["select"], fmt=s["fmt"])
    if kind == "linear":
        return s["linear"](layers.quantize_tokens(s["x"], s["order"], s["select"], s["fmt"]))
    if kind in ("prefill", "qwen"):
        return s["layer"](s["x"])
    if kind == "decode":
        step, cache = s["step"], s["cache"]
        y = step(step.x) if step is not None else s["layer"](s["x"], cache, cache.positions, 0)
        return {"y": y, "pages": cache.pages, "params": cache.scales}
    return s["block"](s["x"], router_logits=s["logits"])[0]


# ------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------

def _quantized_bytes(rows, kp, fmt):
    return rows * (kp // 2 + kp // GROUP[fmt])


def _layer_work(rows, shapes, hidden, fmt):
    """rows through linears [(n, k')]: bf16 activations in and out once, every quantized weight once"""
    return (4 * rows * hidden + sum(_quantized_bytes(n, kp, fmt) for n, kp in shapes),
            sum(2 * rows * n * kp for n, kp in shapes))


def work(case):
    kind, fmt = case["kind"], case["fmt"]
    if kind == "norm":
        rows, k = case["rows"], case["k"]
        return {"bytes": 2 * rows * k + 4 * k + _quantized_bytes(rows, k + case["select"], fmt), "flops": 0}
    if kind == "linear":
        rows, n, k = case["rows"], case["n"], case["k"]
        kp = k + case["select"]
        return {"bytes": 2 * rows * (k + n) + _quantized_bytes(n, kp, fmt), "flops": 2 * rows * n * kp}
    llama = [((HEADS + 2 * KV_HEADS) * HEAD_DIM, HIDDEN + 256), (HIDDEN, HIDDEN + 256), (2 * INTER, HIDDEN + 256),
             (HIDDEN, INTER + 256)]
    if kind in ("prefill", "qwen"):
        b, s = case["batch"], case["seq"]
        if kind == "prefill":
            shapes, hidden, heads = llama, HIDDEN, HEADS
        else:
            kp = Q_HIDDEN + 128
            shapes = [(Q_HIDDEN + 2 * Q_KV_HEADS * HEAD_DIM, kp), (Q_HIDDEN, kp), (2 * Q_INTER, kp), (Q_HIDDEN, Q_INTER + 128)]
            hidden, heads = Q_HIDDEN, Q_HEADS
        nbytes, flops = _layer_work(b * s, shapes, hidden, fmt)
        return {"bytes": nbytes, "flops": flops + 2 * b * heads * s * (s + 1) * HEAD_DIM}      # causal attention
    if kind == "decode":
        b, kv = case["batch"], case["kv"]
        nbytes, flops = _layer_work(b, llama, HIDDEN, fmt)
        nbytes += b * kv * 2 * KV_HEADS * (HEAD_DIM // 2 + 4)                                   # codes and (scale, zero) pairs
        return {"bytes": nbytes, "flops": flops + 4 * b * kv * HEADS * HEAD_DIM}
    pairs = case["tokens"] * TOP_K
    used = min(EXPERTS, pairs)
    kp1, kp2 = HIDDEN + 128, INTER + 128
    weights = used * (_quantized_bytes(2 * INTER, kp1, fmt) + _quantized_bytes(HIDDEN, kp2, fmt))
    return {"bytes": 4 * case["tokens"] * HIDDEN + weights, "flops": 2 * pairs * (2 * INTER * kp1 + HIDDEN * kp2)}


def tolerance(case):
    """norm: the quantizer is exact.  linear: FP4 products sum exactly or nearly so in fp32, in whatever order; what can
    differ is the bf16 rounding of the result (1.7e-3 against 64-bit sums).  Layers with attention in front of a quantizer:
    an attention output one bf16 rounding away moves FP4 codes that lie near a decision point (fp32 attention in place of
    the bf16 flash kernel: 3.0e-2 to 4.4e-2 on a layer's output)."""
    kind = case["kind"]
    if kind == "norm":
        return "exact"
    if kind == "linear":
        return {"rel": 2e-3}
    if kind == "moe":
        return {"rel": 2e-2}
    if kind == "decode":
        return {"rel": 0.12, "differ": 1e-4}
    return {"rel": 0.12}
