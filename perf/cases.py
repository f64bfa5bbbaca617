"""Timing cases of the FP8 linear path: the calls a serving program makes, at the sizes
it makes them.

Three kinds of case, each a dict of plain values:

* ``linear``: one pass through ``LinearMethod.apply`` (activation quantization, product,
  scales, bias) of every projection in ``shapes`` (``"NxK+NxK"``) of every layer.
  ``graph`` cases replay one HIP graph of the whole pass, as a decode loop does; the
  others call the layers one by one, as a prefill does.
* ``moe``: activation quantization and the grouped block-128 product over the experts'
  rows, as one MoE projection runs.
* ``kv``: one write of a batch's keys and values into an FP8 paged cache and the
  dequantizing gather of both planes.

``listed`` holds the sizes of the repository's own configurations; ``draw`` gives others
of the same ranges: 1 to 64 rows for decode, 65 to 8192 for prefill, widths from 1024 to
57344, ragged widths, 1 to 4096 routed tokens, 16 to 65536 cached tokens.
"""

from __future__ import annotations

import math
import os
import sys

import torch
from torch import nn

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), os.pardir, "ayaka-py_amd"))

FP8 = torch.float8_e4m3fn
DEVICE = "cuda"
RECIPES = ("rowwise", "per_tensor_dynamic", "per_tensor_static", "block128", "mxfp8", "w8a16")
CONFIG = {
    "rowwise": {"fp8_recipe": "w8a8_rowwise"},
    "per_tensor_dynamic": {"quant_method": "fp8", "activation_scheme": "dynamic"},
    "per_tensor_static": {"quant_method": "fp8", "activation_scheme": "static"},
    "block128": {"weight_block_size": [128, 128], "scale_format": "float32"},
    "mxfp8": {"quant_algo": "mxfp8"},
    "w8a16": {"quant_algo": "w8a16"},
}
QWEN3_MLP = "3072x1024"
LLAMA3_8B = "6144x4096+4096x4096+28672x4096+4096x14336"
QWEN2_MLP = "37888x3584+3584x18944"
DSV3_DENSE = "18432x7168+7168x18432"
LLAMA3_70B_MLP = "57344x8192+8192x28672"
# The largest listed passes do about this much; drawn ones stay below.
MOST_FLOPS = 8.0e11
MOST_EXPERT_BYTES = 7.6e9


def _linear(name, recipe, m, shapes, *, layers=1, graph=False, dtype="bfloat16", bias=False, block=0):
    case = {"kind": "linear", "recipe": recipe, "m": m, "shapes": shapes, "layers": layers, "graph": graph,
            "dtype": dtype, "bias": bias, "block": block}
    return {"name": name, **case} if name else case


def _moe(name, tokens, topk, experts, n, k):
    case = {"kind": "moe", "tokens": tokens, "topk": topk, "experts": experts, "n": n, "k": k}
    return {"name": name, **case} if name else case


def _kv(name, tokens, heads, dim, dtype="bfloat16", cache="float8_e4m3fn"):
    case = {"kind": "kv", "tokens": tokens, "heads": heads, "dim": dim, "dtype": dtype, "cache": cache}
    return {"name": name, **case} if name else case


def listed():
    return [
        # The smallest call: one MLP projection of a 0.6B model for a batch of 8, called by itself.
        _linear("small_dynamic_m8", "per_tensor_dynamic", 8, QWEN3_MLP),
        # Single-stream decode of an 8B model, weight-only: four layers of a token's graph.
        _linear("decode_w8a16_m1", "w8a16", 1, LLAMA3_8B, layers=4, graph=True),
        # The same for a batch of 16 requests.
        _linear("decode_w8a16_m16", "w8a16", 16, LLAMA3_8B, layers=4, graph=True),
        # Batched decode of DeepSeek-V3's dense layers.
        _linear("decode_block128_m32", "block128", 32, DSV3_DENSE, layers=3, graph=True),
        # A ragged shard: neither the rows nor the widths fill a tile, static scales, fp16, bias.
        _linear("ragged_static_m333", "per_tensor_static", 333, "7392x4096+4096x3696", dtype="float16", bias=True),
        # A chunk of a chunked prefill of a 70B MLP.
        _linear("chunk_mxfp8_m512", "mxfp8", 512, LLAMA3_70B_MLP),
        # Weight-only prefill of an 8B model's layer.
        _linear("prefill_w8a16_m1024", "w8a16", 1024, LLAMA3_8B),
        # Prefill of a 7B MLP with per-token scales and bias.
        _linear("prefill_rowwise_m2048", "rowwise", 2048, QWEN2_MLP, bias=True),
        # A long prefill through the up projection of DeepSeek-V3's dense layers.
        _linear("prefill_block128_m4096", "block128", 4096, "18432x7168"),
        # MoE gate_up while decoding: 64 requests over 256 experts, two rows an expert.
        _moe("moe_decode_t64", 64, 8, 256, 4096, 7168),
        # MoE gate_up while prefilling: 4096 tokens.
        _moe("moe_prefill_t4096", 4096, 8, 256, 4096, 7168),
        # KV cache of a prefill batch: 8 heads x 128.
        _kv("kv_prefill_t32768", 32768, 8, 128),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)) - 1e-9)))))


def _pairs(shapes):
    return [tuple(int(v) for v in s.split("x")) for s in shapes.split("+")]


def _draw_shapes(rng):
    if rng.random() < 0.4:
        return rng.choice((QWEN3_MLP, LLAMA3_8B, QWEN2_MLP, DSV3_DENSE, LLAMA3_70B_MLP))
    hidden, inter = 128 * _log_int(rng, 8, 64), 128 * _log_int(rng, 16, 160)
    return f"{2 * inter}x{hidden}+{hidden}x{inter}"


def draw(rng):
    kind = rng.choice(("decode", "decode", "prefill", "prefill", "ragged", "moe", "kv"))
    dtype = rng.choice(("bfloat16", "bfloat16", "float16"))
    recipe = rng.choice(RECIPES)
    if kind == "decode":
        shapes = _draw_shapes(rng)
        size = sum(n * k for n, k in _pairs(shapes))
        block = 128 if recipe == "w8a16" and rng.random() < 0.25 else 0
        return _linear("", recipe, _log_int(rng, 1, 64), shapes, layers=max(1, min(6, int(6e8 // size))), graph=True,
                       dtype=dtype, block=block)
    if kind == "prefill":
        shapes = _draw_shapes(rng)
        most = MOST_FLOPS / 2 if recipe == "w8a16" else MOST_FLOPS
        m = _log_int(rng, 65, 8192)
        m = min(m, int(most / (2 * sum(n * k for n, k in _pairs(shapes)))))
        block = 128 if recipe == "w8a16" and rng.random() < 0.25 else 0
        return _linear("", recipe, m, shapes, dtype=dtype, bias=rng.random() < 0.3, block=block)
    if kind == "ragged":
        unit = {"block128": 128, "mxfp8": 32}.get(recipe, 16)
        n, k = _log_int(rng, 200, 12000), unit * _log_int(rng, max(1, 256 // unit), 8192 // unit)
        return _linear("", recipe, _log_int(rng, 2, 2048), f"{n}x{k}", dtype=dtype, bias=rng.random() < 0.3)
    if kind == "moe":
        experts = rng.choice((8, 16, 32, 64, 128, 256))
        n, k = 128 * _log_int(rng, 6, 64), 128 * _log_int(rng, 8, 64)
        while experts * n * k > MOST_EXPERT_BYTES:
            experts //= 2
        topk = rng.choice((1, 2, 4, 8))
        tokens = _log_int(rng, 1, 4096)
        tokens = max(1, min(tokens, int(MOST_FLOPS / (2 * topk * n * k))))
        return _moe("", tokens, topk, experts, n, k)
    return _kv("", _log_int(rng, 16, 65536), rng.choice((1, 2, 4, 8, 16)), rng.choice((64, 128, 192, 256)), dtype=dtype,
               cache=rng.choice(("float8_e4m3fn", "float8_e4m3fn", "float8_e5m2")))


# ---------------------------------------------------------------- inputs
def _rows_scale(w):
    return w.abs().amax(dim=1).float().clamp_min(1e-12) / 448.0


def _cast(w):
    return w.clamp_(-448, 448).to(FP8)


def _weight(case, n, k, gen):
    """(e4m3 [N, K] weight, its scales as the checkpoint holds them)."""
    recipe = case["recipe"]
    wf = torch.randn(n, k, generator=gen, device=DEVICE).mul_(0.02)
    if recipe == "mxfp8":
        g = wf.view(n, k // 32, 32)
        e = torch.ceil(torch.log2((g.abs().amax(dim=-1) / 448.0).clamp_min(1e-38))).clamp(-126, 127)
        return _cast(g.div_(torch.exp2(e)[..., None])).view(n, k), (e + 127).to(torch.uint8)
    if recipe == "block128" or case["block"]:
        nb, kb = -(-n // 128), -(-k // 128)
        # blocks of a trained weight differ in magnitude: 10^U(-1, 1)
        wf.mul_(torch.pow(10.0, 2 * torch.rand(nb, kb, generator=gen, device=DEVICE) - 1)
                .repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :k])
        pad = torch.zeros(nb * 128, kb * 128, device=DEVICE)
        pad[:n, :k] = wf
        s = pad.view(nb, 128, kb, 128).abs_().amax(dim=(1, 3)).clamp_min_(1e-12) / 448.0
        del pad
        return _cast(wf.div_(s.repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :k])), s
    if recipe.startswith("per_tensor"):
        s = (wf.abs().amax() / 448.0).expand(n).contiguous()
    else:
        s = _rows_scale(wf)
    return _cast(wf.div_(s[:, None])), s


def _activation(m, k, gen, dtype):
    """N(0, 1) with 1% of the channels twenty times larger, as LLM activations are."""
    x = torch.randn(m, k, generator=gen, device=DEVICE)
    loud = torch.randperm(k, generator=gen, device=DEVICE)[: max(1, k // 100)]
    x[:, loud] *= 20.0
    return x.to(getattr(torch, dtype))


def _linear_inputs(case, seed):
    """Activation and bias of every projection, and an iterator over the layers' weights."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    pairs = _pairs(case["shapes"])
    xs = [_activation(case["m"], k, gen, case["dtype"]) for _, k in pairs]
    biases = [torch.randn(n, generator=gen, device=DEVICE).to(xs[0].dtype) if case["bias"] else None for n, _ in pairs]
    weights = (_weight(case, n, k, gen) for _ in range(case["layers"]) for n, k in pairs)
    return xs, biases, weights


def _input_scale(x):
    return (x.abs().amax().float() / 448.0).reshape(())


def _make_layer(case, x, w, s):
    from ayaka.layers.linear.fp8 import FP8Config

    if case["block"]:
        config = FP8Config("w8a16", scale_dtype=torch.float32, weight_block=(128, 128))
    else:
        config = FP8Config.from_config(CONFIG[case["recipe"]])
    method = config.get_quant_method(None, "model.layers.0.mlp.proj")
    layer = nn.Module()
    method.create_weights(layer, output_partition_sizes=[w.shape[0]], input_size_per_partition=w.shape[1], device=DEVICE)
    layer.weight.data.copy_(w)
    param = layer.weight_scale_inv if case["recipe"] == "block128" else layer.weight_scale
    param.weight_loader(layer, param, s)
    if case["recipe"] == "per_tensor_static":
        layer.input_scale.weight_loader(layer, layer.input_scale, _input_scale(x))
    method.process_weights_after_loading(layer)
    return method, layer


def _moe_inputs(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    experts, n, k = case["experts"], case["n"], case["k"]
    # routers are not uniform: log-normal expert popularity
    popularity = torch.exp(0.5 * torch.randn(experts, generator=gen, device=DEVICE))
    picks = torch.multinomial(popularity, case["tokens"] * case["topk"], replacement=True, generator=gen)
    counts = torch.bincount(picks, minlength=experts)
    offsets = counts.cumsum(0) - counts
    x = _activation(case["tokens"] * case["topk"], k, gen, "bfloat16")
    b = torch.empty(experts, n, k, dtype=FP8, device=DEVICE)
    for e in range(experts):
        b[e] = (torch.randn(n, k, generator=gen, device=DEVICE, dtype=torch.bfloat16) * 100).clamp_(-448, 448).to(FP8)
    sb = torch.pow(10.0, 2 * torch.rand(experts, n // 128, k // 128, generator=gen, device=DEVICE) - 1) * 2e-4
    return x, b, sb, counts, offsets


KV_PAGE = 16


def _kv_inputs(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    t, heads, dim = case["tokens"], case["heads"], case["dim"]
    key, value = (torch.randn(t, heads, dim, generator=gen, device=DEVICE).to(getattr(torch, case["dtype"]))
                  for _ in range(2))
    used = -(-t // KV_PAGE)
    pages = max(64, 2 * used)
    table = torch.randperm(pages, generator=gen, device=DEVICE)[:used]  # pages as the allocator handed them out
    pos = torch.arange(t, device=DEVICE)
    slots = table[pos // KV_PAGE] * KV_PAGE + pos % KV_PAGE
    return key, value, pages, slots


def prepare(case, seed):
    if case["kind"] == "linear":
        xs, biases, weights = _linear_inputs(case, seed)
        calls = []
        for i, (w, s) in enumerate(weights):
            j = i % len(xs)
            method, layer = _make_layer(case, xs[j], w, s)
            calls.append((method.apply, layer, xs[j], biases[j]))
            del w, s
        state = {"calls": calls}
        if case["graph"]:
            stream = torch.cuda.Stream()
            stream.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(stream):
                state["outputs"] = _apply_all(calls)
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=stream):
                    state["outputs"] = _apply_all(calls)
            torch.cuda.current_stream().wait_stream(stream)
            state["graph"] = graph
        return state
    if case["kind"] == "moe":
        x, b, sb, counts, offsets = _moe_inputs(case, seed)
        experts, n, k = case["experts"], case["n"], case["k"]
        sizes = torch.stack([counts, torch.full_like(counts, n), torch.full_like(counts, k)], 1).to(torch.int32)
        return {
            "moe": True, "x": x, "b": b, "sb": sb, "sizes": sizes, "offsets": offsets.to(torch.int32),
            "out": torch.zeros(x.shape[0], n, dtype=x.dtype, device=DEVICE),
            "tables": [torch.empty(experts, dtype=torch.int64, device=DEVICE) for _ in range(5)],
            "strides": [torch.full((experts,), v, dtype=torch.int64, device=DEVICE) for v in (k, k, n)],
            "layouts": [torch.empty(experts, 5, dtype=torch.int32, device=DEVICE) for _ in range(2)],
            "workspace": torch.empty(1, dtype=torch.uint8, device=DEVICE),
        }
    key, value, pages, slots = _kv_inputs(case, seed)
    shape = (pages, KV_PAGE, case["heads"], case["dim"])
    cache = getattr(torch, case["cache"])
    caches = [torch.zeros(shape, dtype=torch.uint8, device=DEVICE).view(cache) for _ in range(2)]
    return {"key": key, "value": value, "slots": slots, "caches": caches,
            "gathered": [torch.zeros_like(key) for _ in range(2)]}


def _apply_all(calls):
    return [apply(layer, x, bias) for apply, layer, x, bias in calls]


KV_SCALE = 0.5


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    if "calls" in state:
        return _apply_all(state["calls"])
    if "moe" in state:
        from ayaka.kernel.hip import fp8_blockwise_scaled_grouped_mm, per_token_group_quant_fp8

        q, scale = per_token_group_quant_fp8(state["x"], 128)
        fp8_blockwise_scaled_grouped_mm(state["out"], *state["tables"], q, state["b"], scale, state["sb"],
                                        *state["strides"], *state["layouts"], state["sizes"], state["offsets"],
                                        state["workspace"])
        return state["out"]
    from ayaka.kernel.hip import gather_cache, write_kv

    caches, slots = state["caches"], state["slots"]
    write_kv(state["key"], state["value"], *caches, slots, 1.0 / KV_SCALE, 1.0 / KV_SCALE)
    for cache, out in zip(caches, state["gathered"]):
        gather_cache(cache, slots, out, KV_SCALE, True)
    return [c.view(torch.uint8) for c in caches] + state["gathered"]


def work(case):
    if case["kind"] == "linear":
        m, total, flops = case["m"], 0, 0
        for n, k in _pairs(case["shapes"]):
            scales = {"mxfp8": n * k // 32, "block128": 4 * -(-n // 128) * -(-k // 128)}.get(case["recipe"], 4 * n)
            total += n * k + scales + 2 * m * k + 2 * m * n + (2 * n if case["bias"] else 0)
            flops += 2 * m * n * k
        return {"bytes": total * case["layers"], "flops": flops * case["layers"]}
    if case["kind"] == "moe":
        rows, e, n, k = case["tokens"] * case["topk"], case["experts"], case["n"], case["k"]
        hit = e * (1 - (1 - 1 / e) ** rows)  # experts that a uniform router reaches
        return {"bytes": hit * (n * k + 4 * (n // 128) * (k // 128)) + 2 * rows * (n + k), "flops": 2 * rows * n * k}
    size = case["tokens"] * case["heads"] * case["dim"]
    return {"bytes": 2 * size * (2 + 1) + 2 * size * (1 + 2) + 3 * 8 * case["tokens"], "flops": 0}


def tolerance(case):
    if case["kind"] == "kv":
        return "exact"
    # Products of 8-bit or 16-bit operands summed in fp32 and rounded once to a 16-bit
    # output. Against 64 bits the results are 1.6e-3 (bf16) and 2.1e-4 (fp16) off, the
    # rounding of the output, and 2.3e-3 to 2.8e-3 / 3e-4 where a weight-only product rounds the
    # dequantized weight as well, which an implementation may or may not do: about four
    # times that, and four units of the output type at a single value.
    if case.get("dtype") == "float16":
        return {"rel": 1.2e-3, "max": 4e-3}
    return {"rel": 9e-3, "max": 3.2e-2}


# ---------------------------------------------------------------- 64-bit results
def _over_448(amax):
    """amax / 448 in fp32, correctly rounded (torch divides by a number on the GPU as a
    product with its reciprocal, which moves scales, and with them codes, by an ulp)."""
    return amax / torch.full_like(amax, 448.0)


def _e8m0(codes):
    return torch.exp2(codes.double() - 127.0) * (codes != 0)


def _dequantized_weight(case, w, s):
    n, k = w.shape
    w = w.double()
    if case["recipe"] == "mxfp8":
        return w.view(n, k // 32, 32).mul_(_e8m0(s)[..., None]).view(n, k)
    if case["recipe"] == "block128" or case["block"]:
        return w.mul_(s.double().repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :k])
    return w.mul_(s.double()[:, None])


def _group_quantized(x, group):
    """Dynamic fp8 quantization per (row, group), decoded: codes as the fp32 rule gives them."""
    g = x.float().view(x.shape[0], -1, group)
    s = _over_448(g.abs().amax(dim=-1).clamp_min(1e-10))
    q = (g / s[..., None]).clamp(-448, 448).to(FP8)
    return (q.double() * s.double()[..., None]).view(x.shape)


def _quantized_activation(case, x):
    recipe, m = case["recipe"], x.shape[0]
    if recipe == "mxfp8":
        g = x.float().view(m, -1, 32)
        amax = g.abs().amax(dim=-1)
        e = torch.ceil(torch.log2(_over_448(amax).clamp_min(1e-38))).clamp(-126, 127)
        q = (g / torch.exp2(e)[..., None]).clamp(-448, 448).to(FP8).double()
        return (q * torch.exp2(e.double())[..., None]).view(x.shape)
    if recipe == "w8a16" or m == 1:
        return x.double()
    if recipe == "block128":
        return _group_quantized(x, 128)
    if recipe == "per_tensor_static":
        s = _input_scale(x)
        return (x.float() / s).clamp(-448, 448).to(FP8).double() * s.double()
    return _group_quantized(x, x.shape[1])


def exact(case, seed):
    if case["kind"] == "linear":
        xs, biases, weights = _linear_inputs(case, seed)
        outs = []
        for i, (w, s) in enumerate(weights):
            j = i % len(xs)
            a = _quantized_activation(case, xs[j])
            y = torch.empty(a.shape[0], w.shape[0], dtype=torch.float64, device=DEVICE)
            for n0 in range(0, w.shape[0], 8192):  # in slices: 64-bit weights are large; N0 a multiple of 128
                rows = slice(n0, min(n0 + 8192, w.shape[0]))
                scales = s[n0 // 128:-(-rows.stop // 128)] if case["recipe"] == "block128" or case["block"] else s[rows]
                y[:, rows] = a @ _dequantized_weight(case, w[rows], scales).t()
            if biases[j] is not None:
                y += biases[j].double()
            # One row of a weight-only product comes back without its row dimension.
            outs.append(y.view(-1) if case["m"] == 1 and case["recipe"] == "w8a16" else y)
        return outs
    if case["kind"] == "moe":
        x, b, sb, counts, offsets = _moe_inputs(case, seed)
        a = _group_quantized(x, 128)
        y = torch.zeros(x.shape[0], case["n"], dtype=torch.float64, device=DEVICE)
        for e, (off, count) in enumerate(zip(offsets.tolist(), counts.tolist())):
            if count:
                w = b[e].double().mul_(sb[e].double().repeat_interleave(128, 0).repeat_interleave(128, 1))
                y[off:off + count] = a[off:off + count] @ w.t()
        return y
    key, value, _, _ = _kv_inputs(case, seed)
    cache = getattr(torch, case["cache"])
    limit = torch.finfo(cache).max
    decoded = [(p.float() / KV_SCALE).clamp(-limit, limit).to(cache).double() * KV_SCALE for p in (key, value)]
    return [None, None] + decoded
