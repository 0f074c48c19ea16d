"""Performance cases: the work a user of this package has it do, each through
its public entry points.

A case is a dict of plain values.  ``op`` names the path:

* ``linear``    ``QuantLinear.forward`` on ``[M, K]`` activations;
* ``mlp``       a SwiGLU MLP block: RMSNorm + gate|up + SwiGLU, then down;
* ``chain``     the projections of decoder layers as one ``DecodeChain``;
* ``step``      a whole batch-1 token step replayed from a HIP graph;
* ``attention`` one token's grouped-query attention over a KV cache;
* ``dequant``   a packed weight expanded to dense fp16;
* ``quantize``  a dense weight packed to INT4 on the GPU.

``layout`` is ``packed`` (the checkpoint format) or ``strip`` (the decode
layout ``QuantLinear.prepare_decode`` converts to).  Shapes are those of the
8B-shaped model of :mod:`nibblegemm_amd.decode_step` and of the benchmark
sweeps, plus generic ragged ones.
"""
import math

import torch

from nibblegemm_amd import QuantizedWeight, QuantLinear, dequant, matmul
from nibblegemm_amd.chain import DecodeChain, chain_strip_cols, stage
from nibblegemm_amd.decode_step import GlueDecodeStep
from nibblegemm_amd.glue import attention_decode, rope_tables
from nibblegemm_amd.ops import rmsnorm_matmul, strip_major_cols
from nibblegemm_amd.quant import quantize_device

EPS = 1e-5
HEADS, KV_HEADS, HEAD_DIM = 32, 8, 128
#: Nibble slot of logical offset k within a packed word (the checkpoint format).
SLOTS = (0, 4, 1, 5, 2, 6, 3, 7)
SWIGLU_BLOCK = 16  # columns per gate / up block of an interleaved weight


def listed():
    return [
        # One k or v projection for one token, called eagerly: the smallest
        # call, where the launch and the call's own latency are everything.
        {"name": "kv_proj_b1", "op": "linear", "M": 1, "K": 4096, "N": 1024, "g": 128,
         "layout": "packed", "bias": False},
        # The down projection of a small decode batch on weights converted for
        # decoding, with a bias.
        {"name": "down_b8_strip", "op": "linear", "M": 8, "K": 14336, "N": 4096, "g": 128,
         "layout": "strip", "bias": True},
        # Batch-1 decoding as a serving loop runs it: four layers of the
        # 8B-shaped model, norms and attention over 1024 tokens included,
        # replayed from a graph.
        {"name": "step_ctx1024", "op": "step", "layers": 4, "ctx": 1024, "g": 128},
        # The same layers' projections in one persistent launch on the packed
        # checkpoint weights (the reference's decode-step benchmark, which
        # feeds every projection a fixed activation).
        {"name": "chain_8_layers", "op": "chain", "layers": 8, "hidden": 4096, "inter": 14336,
         "kv": 1024, "g": 128},
        # One MLP block of a batched decode step.
        {"name": "mlp_b32", "op": "mlp", "M": 32, "hidden": 4096, "inter": 14336, "g": 128},
        # A larger decode batch, or a short prompt, on a 70B-shaped attention
        # projection.
        {"name": "attn_proj_b96", "op": "linear", "M": 96, "K": 8192, "N": 8192, "g": 128,
         "layout": "packed", "bias": False},
        # Prefill of an ordinary prompt: the gate or up projection.
        {"name": "gate_512", "op": "linear", "M": 512, "K": 4096, "N": 14336, "g": 128,
         "layout": "packed", "bias": False},
        # Prefill of a long prompt, a whole MLP block: the largest case.
        {"name": "mlp_2048", "op": "mlp", "M": 2048, "hidden": 4096, "inter": 14336, "g": 128},
        # A model with groups of 64, an output width that is no multiple of 4
        # and a prompt length that fills no tile.
        {"name": "ragged_1000", "op": "linear", "M": 1000, "K": 5504, "N": 4102, "g": 64,
         "layout": "packed", "bias": True},
        # Attention of one token late in a long conversation.
        {"name": "attention_8192", "op": "attention", "ctx": 8192, "heads": HEADS,
         "kv_heads": KV_HEADS},
        # A weight expanded for a library that wants it dense.
        {"name": "dequant_up", "op": "dequant", "K": 4096, "N": 14336, "g": 128},
        # A weight of an fp16 checkpoint quantised while a model is loaded.
        {"name": "quantize_up", "op": "quantize", "K": 4096, "N": 14336, "g": 128,
         "dtype": "float16"},
    ]


# ---------------------------------------------------------------- drawn cases

#: Multiply-adds of the largest listed case's largest product.
_MAX_MACS = 2048 * 4096 * 28672


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, multiple):
    """A width in [lo, hi]: often a multiple of 128, else only of ``multiple``."""
    m = rng.choice([128, 128, multiple])
    return max(m, _log_int(rng, lo, hi) // m * m)


def draw(rng):
    op = rng.choice(["linear"] * 6 + ["mlp", "mlp", "chain", "step", "attention", "dequant",
                                      "quantize"])
    g = rng.choice([128, 128, 64])
    if op == "linear":
        layout = rng.choice(["packed", "packed", "strip"])
        M = _log_int(rng, 1, 4096)
        K = _log_int(rng, 1024, 14336) // g * g
        # strips of 64, 32 or 16 columns; the decode kernels take multiples of
        # 4, the prefill kernels of 2
        N = _width(rng, 1024, 14336, 64 if layout == "strip" else 4 if M <= 8 else 2)
        M = max(1, min(M, _MAX_MACS // (K * N)))
        return {"op": op, "M": M, "K": K, "N": N, "g": g, "layout": layout,
                "bias": rng.random() < 0.5}
    if op == "mlp":
        return {"op": op, "M": _log_int(rng, 1, 2048), "hidden": _log_int(rng, 1024, 4096) // 128 * 128,
                "inter": _log_int(rng, 2048, 14336) // 128 * 128, "g": g}
    if op == "chain":
        return {"op": op, "layers": rng.randint(1, 8), "hidden": _log_int(rng, 1024, 4096) // 256 * 256,
                "inter": _log_int(rng, 2048, 14336) // 256 * 256,
                "kv": rng.choice([512, 1024]), "g": 128}
    if op == "step":
        return {"op": op, "layers": rng.randint(1, 4), "ctx": _log_int(rng, 2, 8192), "g": g}
    if op == "attention":
        kv = rng.choice([2, 4, 8])
        return {"op": op, "ctx": _log_int(rng, 64, 32768), "heads": kv * rng.choice([1, 4, 8]),
                "kv_heads": kv}
    K = _log_int(rng, 1024, 14336) // g * g
    case = {"op": op, "K": K, "N": _width(rng, 1024, 14336, 4), "g": g}
    if op == "quantize":
        case["dtype"] = rng.choice(["float16", "float32"])
    return case


# --------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _weight(gen, K, N, g):
    """A packed weight with the codes and scales that round-to-nearest
    quantisation of ``randn * 0.02`` has: the largest of a group's g values is
    2.4 to 2.7 standard deviations, which becomes code 7."""
    spread = 7.0 / (2.7 if g == 128 else 2.4)
    words = torch.zeros((K // 8, N), dtype=torch.int32, device="cuda")
    for slot in SLOTS:
        codes = torch.randn((K // 8, N), generator=gen, device="cuda").mul_(spread).round_()
        words |= (codes.clamp_(-7, 7) + 8).to(torch.int32) << (4 * slot)
    scales = (0.02 / spread) * (1 + 0.12 * torch.randn((K // g, N), generator=gen, device="cuda"))
    return QuantizedWeight(words, scales.clamp_(min=1e-3).to(torch.float16), g, K, N)


def _act(gen, M, K):
    return torch.randn((M, K), generator=gen, device="cuda").to(torch.float16)


def _norm_weight(gen, n):
    return (1 + 0.05 * torch.randn(n, generator=gen, device="cuda")).to(torch.float16)


def _layer_shapes(case):
    h, inter, kv = case["hidden"], case["inter"], case["kv"]
    return [("qkv", h, h + 2 * kv), ("o", h, h), ("gate_up", h, 2 * inter), ("down", inter, h)]


def _prepare_linear(case, gen):
    qw = _weight(gen, case["K"], case["N"], case["g"])
    bias = None
    if case["bias"]:
        bias = torch.randn(case["N"], generator=gen, device="cuda").to(torch.float16)
    x = _act(gen, case["M"], case["K"])
    layer = QuantLinear(qw, bias)
    if case["layout"] == "strip" and strip_major_cols(qw.K, qw.N, qw.group_size):
        layer.prepare_decode()
    return {"x": x, "qw": qw, "bias": bias, "layer": layer}


def _prepare_mlp(case, gen):
    h, inter, g = case["hidden"], case["inter"], case["g"]
    return {"x": _act(gen, case["M"], h), "norm": _norm_weight(gen, h),
            "gate_up": _weight(gen, h, 2 * inter, g),  # interleaved gate|up blocks
            "down": _weight(gen, inter, h, g)}


def _chain_inputs(case, gen):
    layers = [{name: _weight(gen, K, N, case["g"]) for name, K, N in _layer_shapes(case)}
              for _ in range(case["layers"])]
    acts = {K: _act(gen, 1, K) for K in sorted({case["hidden"], case["inter"]})}
    return layers, acts


def _prepare_chain(case, gen):
    layers, acts = _chain_inputs(case, gen)
    stages = [stage(acts[w.K], w, strip_cols=chain_strip_cols(w.K, w.N, w.group_size))
              for layer in layers for w in layer.values()]
    return {"chain": DecodeChain(stages)}


def _step_inputs(case, gen, seed):
    h, inter, kv, g = 4096, 14336, 1024, case["g"]
    layers = [{"qkv": _weight(gen, h, h + 2 * kv, g), "o": _weight(gen, h, h, g),
               "gate_up_swiglu": _weight(gen, h, 2 * inter, g), "down": _weight(gen, inter, h, g)}
              for _ in range(case["layers"])]
    return GlueDecodeStep(layers, pos=case["ctx"] - 1, seed=int(seed) + 1)


def _prepare_step(case, gen, seed):
    step = _step_inputs(case, gen, seed)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return {"step": step, "graph": graph, "out": out}


def _prepare_attention(case, gen):
    heads, kv, ctx = case["heads"], case["kv_heads"], case["ctx"]
    caches = [torch.randn((kv, ctx, HEAD_DIM), generator=gen, device="cuda").to(torch.float16)
              for _ in range(2)]
    return {"qkv": _act(gen, 1, (heads + 2 * kv) * HEAD_DIM), "k": caches[0], "v": caches[1],
            "pos": ctx - 1, "rope": rope_tables(ctx)}


def prepare(case, seed):
    gen = _gen(seed)
    op = case["op"]
    if op == "linear":
        state = _prepare_linear(case, gen)
        del state["qw"], state["bias"]
    elif op == "mlp":
        state = _prepare_mlp(case, gen)
    elif op == "chain":
        state = _prepare_chain(case, gen)
    elif op == "step":
        state = _prepare_step(case, gen, seed)
    elif op == "attention":
        state = _prepare_attention(case, gen)
    elif op == "dequant":
        state = {"qw": _weight(gen, case["K"], case["N"], case["g"])}
    else:
        state = {"W": _dense(case, gen), "g": case["g"]}
    state["op"] = op
    return state


def _dense(case, gen):
    W = torch.randn((case["K"], case["N"]), generator=gen, device="cuda") * 0.02
    return W.to(getattr(torch, case["dtype"]))


# ------------------------------------------------------------------- one pass

def run(state):
    op = state["op"]
    if op == "linear":
        return state["layer"](state["x"])
    if op == "mlp":
        g = rmsnorm_matmul(state["x"], state["norm"], state["gate_up"], EPS, swiglu=True)
        return [g, matmul(g, state["down"])]
    if op == "chain":
        state["chain"].run()
        return state["chain"].outputs()
    if op == "step":
        state["graph"].replay()
        return [state["out"]] + [c for pair in state["step"].caches for c in pair]
    if op == "attention":
        out = attention_decode(state["qkv"], state["k"], state["v"], state["pos"], state["rope"])
        return [out, state["k"], state["v"]]
    if op == "dequant":
        return dequant(state["qw"])
    qw = quantize_device(state["W"], state["g"])
    return [qw.qweight, qw.scales]


# ------------------------------------------- what a pass cannot do without

def _wbytes(K, N, g):
    return K * N // 2 + K // g * N * 2


def work(case):
    op = case["op"]
    if op == "linear":
        M, K, N, g = case["M"], case["K"], case["N"], case["g"]
        return {"bytes": _wbytes(K, N, g) + 2 * M * (K + N) + (2 * N if case["bias"] else 0),
                "flops": 2 * M * K * N}
    if op == "mlp":
        M, h, inter, g = case["M"], case["hidden"], case["inter"], case["g"]
        return {"bytes": _wbytes(h, 2 * inter, g) + _wbytes(inter, h, g) + 2 * h
                + 2 * M * (2 * h + inter), "flops": 6 * M * h * inter}
    if op == "chain":
        shapes = _layer_shapes(case)
        L = case["layers"]
        return {"bytes": L * sum(_wbytes(K, N, case["g"]) + 2 * N for _, K, N in shapes)
                + 2 * (case["hidden"] + case["inter"]),
                "flops": L * sum(2 * K * N for _, K, N in shapes)}
    if op == "step":
        shapes = _layer_shapes({"hidden": 4096, "inter": 14336, "kv": 1024})
        cache = 2 * KV_HEADS * case["ctx"] * HEAD_DIM * 2
        L = case["layers"]
        return {"bytes": L * (sum(_wbytes(K, N, case["g"]) for _, K, N in shapes) + cache
                              + 2 * 2 * 4096) + 2 * 2 * 4096,
                "flops": L * (sum(2 * K * N for _, K, N in shapes)
                              + 4 * HEADS * case["ctx"] * HEAD_DIM)}
    if op == "attention":
        heads, kv, ctx = case["heads"], case["kv_heads"], case["ctx"]
        return {"bytes": 4 * kv * ctx * HEAD_DIM + 4 * heads * HEAD_DIM + 8 * kv * HEAD_DIM,
                "flops": 4 * heads * ctx * HEAD_DIM}
    K, N, g = case["K"], case["N"], case["g"]
    if op == "dequant":
        return {"bytes": _wbytes(K, N, g) + 2 * K * N, "flops": 0}
    size = 2 if case["dtype"] == "float16" else 4
    return {"bytes": size * K * N + _wbytes(K, N, g), "flops": 0}


def tolerance(case):
    """About four times the differences between the paths and ``exact`` (or
    between two orders of summation): outputs are fp16, so a result is off by
    up to half an ulp of it (3e-4 of it, on average), and each further
    rounding to fp16 on the way (the dequantised weight of the prefill
    kernels, an MLP's middle, a decoder layer's activations) adds as much."""
    op = case["op"]
    if op in ("dequant", "quantize"):
        return "exact"
    if op == "step":
        return {"rel": 5e-3, "max": 3e-2}
    if op == "mlp":
        return {"rel": 2.5e-3, "max": 1.2e-2}
    return {"rel": 1e-3, "max": 5e-3}


# ----------------------------------------------- the same in 64-bit arithmetic

def _dense64(qw):
    """``(code - 8) * scale`` in float64, ``[K, N]``."""
    out = torch.empty((qw.K // 8, 8, qw.N), dtype=torch.float64, device="cuda")
    for k, slot in enumerate(SLOTS):
        out[:, k] = ((qw.qweight >> (4 * slot)) & 15).to(torch.float64) - 8
    out = out.view(qw.K // qw.group_size, qw.group_size, qw.N)
    out *= qw.scales.to(torch.float64)[:, None, :]
    return out.view(qw.K, qw.N)


def _mm64(x, qw):
    return x.double() @ _dense64(qw)


def _rms64(x, w):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _swiglu64(y):
    v = y.view(y.shape[0], -1, 2, SWIGLU_BLOCK)
    return (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(y.shape[0], -1)


def _rotate64(x, rope, pos):
    cos, sin = (t[pos].double() for t in rope)
    a, b = x[..., :HEAD_DIM // 2], x[..., HEAD_DIM // 2:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _attention64(qkv, k_cache, v_cache, pos, rope, heads, kv):
    """Output and the caches with the token's rows written, in float64."""
    q, k, v = qkv.double().view(-1, HEAD_DIM).split([heads, kv, kv])
    k_cache, v_cache = k_cache.double(), v_cache.double()
    k_cache[:, pos], v_cache[:, pos] = _rotate64(k, rope, pos), v
    q = _rotate64(q, rope, pos).view(kv, heads // kv, HEAD_DIM)
    s = q @ k_cache[:, :pos + 1].transpose(1, 2).contiguous() / math.sqrt(HEAD_DIM)
    out = torch.softmax(s, -1) @ v_cache[:, :pos + 1]
    return out.reshape(1, heads * HEAD_DIM), k_cache, v_cache


def exact(case, seed):
    gen = _gen(seed)
    op = case["op"]
    if op == "linear":
        s = _prepare_linear({**case, "layout": "packed"}, gen)
        y = _mm64(s["x"], s["qw"])
        return y if s["bias"] is None else y + s["bias"].double()
    if op == "mlp":
        s = _prepare_mlp(case, gen)
        g = _swiglu64(_mm64(_rms64(s["x"], s["norm"]), s["gate_up"]))
        return [g, _mm64(g, s["down"])]
    if op == "chain":
        layers, acts = _chain_inputs(case, gen)
        return [_mm64(acts[w.K], w) for layer in layers for w in layer.values()]
    if op == "step":
        st = _step_inputs(case, gen, seed)
        h, caches = st.x.double(), []
        for layer, (w_attn, w_ffn), (kc, vc) in zip(st.layers, st.norms, st.caches):
            qkv = _mm64(_rms64(h, w_attn), layer["qkv"])
            att, k64, v64 = _attention64(qkv, kc, vc, st.pos, st.rope, HEADS, KV_HEADS)
            caches += [k64, v64]
            h = h + _mm64(att, layer["o"])
            h = h + _mm64(_swiglu64(_mm64(_rms64(h, w_ffn), layer["gate_up_swiglu"])),
                          layer["down"])
        return [h] + caches
    if op == "attention":
        s = _prepare_attention(case, gen)
        return list(_attention64(s["qkv"], s["k"], s["v"], s["pos"], s["rope"], case["heads"],
                                 case["kv_heads"]))
    if op == "dequant":
        return _dense64(_weight(gen, case["K"], case["N"], case["g"]))
    groups = _dense(case, gen).double().view(-1, case["g"], case["N"])
    return [None, groups.abs().amax(1) / 7]
