"""Performance cases: what a program that serves a language model's linear layers has this package do.

A case names one call pattern and its sizes:

  kind "linear"  ``QuantLinear``'s forward, row-major or pre-packed weights, with or without bias and residual
  kind "gated"   ``torch.ops.awesome_fusion.bfaintb_gemm[_prepacked]`` with the SiLU-gate epilogue (a gated MLP's first half)
  kind "abi"     ``gemm`` / ``gemm_prepacked`` (the C ABI) into the caller's own output with the caller's own workspace
  kind "block"   the four linear layers of a decoder block, captured once in a HIP graph and replayed (a decode step)
  kind "load"    ``QuantLinear.from_float`` and ``prepack``: a checkpoint's bf16 weight to packed codes

m rows of activations, n output columns (of the weights), k inputs; ``bits`` and ``group`` as everywhere in the package.
Activations are N(0, 1); weights are normally distributed and quantised by the package's own absmax quantiser, which is what a
checkpoint goes through.
"""
import math

import torch

import awesome_fusion_amd as af
import awesome_fusion_amd.torch_op as top

_LARGEST_FLOPS = 2 * 2048 * 28672 * 8192     # no drawn case does more
_LARGEST_WEIGHTS = 28672 * 8192
_LARGEST_LOAD = 11008 * 4096


def _case(name, kind, m, n, k, bits, group=0, packed=False, bias=False, residual=False):
    return {"name": name, "kind": kind, "m": m, "n": n, "k": k, "bits": bits, "group": group, "packed": packed, "bias": bias, "residual": residual}


def listed():
    return [
        # one token through a square projection: the headline decode shape, called as a C-ABI user calls it
        _case("abi_m1_4096x4096_int8", "abi", 1, 4096, 4096, 8),
        # a small head of ragged size on a few rows (a classifier, a router): latency and launch overhead, partial tiles
        _case("linear_m3_1040x1000_int8_bias", "linear", 3, 1040, 1000, 8, bias=True),
        # small-batch decode through an MLP up-projection
        _case("linear_m4_11008x4096_int8_bias", "linear", 4, 11008, 4096, 8, bias=True),
        # batched decode on a large model's MLP, 4-bit groupwise codes packed at load time
        _case("linear_m16_28672x8192_int4_packed", "linear", 16, 28672, 8192, 4, 128, packed=True),
        # the output layer of a language model, one token
        _case("abi_m1_128256x4096_int8", "abi", 1, 128256, 4096, 8),
        # gated MLP front half in batched decode, 4-bit groupwise, interleaved (gate, up) columns
        _case("gated_m32_22016x4096_int4", "gated", 32, 22016, 4096, 4, 128),
        # one decode step of a decoder block for 8 sequences, replayed from a graph (hidden 4096, MLP 11008)
        _case("block_m8_4096_11008_int8", "block", 8, 11008, 4096, 8),
        # many concurrent sequences through an MLP down-projection with the residual stream added
        _case("linear_m96_4096x11008_int8_residual", "linear", 96, 4096, 11008, 8, residual=True),
        # a prompt of odd length, packed 4-bit codes
        _case("linear_m577_13824x5120_int4_packed", "linear", 577, 13824, 5120, 4, 128, packed=True),
        # the headline prefill shape
        _case("abi_m4096_4096x4096_int8", "abi", 4096, 4096, 4096, 8),
        # a long prompt through a large model's MLP: the largest
        _case("linear_m2048_28672x8192_int4", "linear", 2048, 28672, 8192, 4, 128),
        # loading: quantise and pack one layer of a checkpoint
        _case("load_11008x4096_int4", "load", 1, 11008, 4096, 4, 128, packed=True),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(rng, lo, hi, step):
    return max(step, _log_uniform(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(("linear",) * 6 + ("abi",) * 3 + ("gated",) * 2 + ("block", "load"))
    while True:
        bits = rng.choice((8, 4))
        group = rng.choice((0, 128)) if bits == 8 else rng.choice((128, 128, 64, 0))
        packed = rng.random() < 0.5
        k = _multiple(rng, 1000, 16384, 128 if packed or group else 8)
        n = _multiple(rng, 1024, 131072 if kind == "abi" else 32768, 16)
        m = _log_uniform(rng, 1, 4096)
        bias, residual = rng.random() < 0.3, rng.random() < 0.3
        if kind == "block":  # n is the MLP's width: a decode step of a batch
            m, k, n = _log_uniform(rng, 1, 64), _multiple(rng, 1024, 4096, 128), _multiple(rng, 2048, 11008, 128)
            bias = residual = False
        elif kind == "load":
            m, residual = 1, False
        elif kind == "gated":
            bias = residual = False
        if kind == "load" and n * k > _LARGEST_LOAD:
            continue
        if n * k <= _LARGEST_WEIGHTS and 2 * m * n * k <= _LARGEST_FLOPS:
            c = _case("", kind, m, n, k, bits, group, packed, bias, residual)
            del c["name"]
            return c


def _block_shapes(case):
    """(n, k) of a decoder block's projections: query-key-value, output, gate and up, down."""
    h, f = case["k"], case["n"]
    return (3 * h, h), (h, h), (2 * f, h), (h, f)


def _rng(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.bfloat16)


def _float_linear(g, n, k, bias):
    lin = torch.nn.utils.skip_init(torch.nn.Linear, k, n, bias=bias, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        lin.weight.normal_(0.0, k ** -0.5, generator=g)
        if bias:
            lin.bias.normal_(0.0, 0.1, generator=g)
    return lin.requires_grad_(False)


def _quant_linear(g, n, k, case):
    layer = top.QuantLinear.from_float(_float_linear(g, n, k, case["bias"]), case["bits"], case["group"])
    if case["packed"]:
        layer.prepack()
    return layer.eval().requires_grad_(False)


def _workspace(nbytes):
    if nbytes == 0:
        return None
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    af.workspace_init(ws)
    return ws


def prepare(case, seed):
    g = _rng(seed)
    m, n, k, bits, group = case["m"], case["n"], case["k"], case["bits"], case["group"]
    if case["kind"] == "load":
        return {"case": case, "linear": _float_linear(g, n, k, case["bias"])}
    if case["kind"] == "block":
        return _prepare_block(g, case)
    x = _normal(g, m, k)
    layer = _quant_linear(g, n, k, case)
    state = {"case": case, "x": x, "layer": layer, "residual": _normal(g, m, n) if case["residual"] else None}
    if case["kind"] == "abi":
        find = af.prepacked_workspace_bytes if case["packed"] else af.workspace_bytes
        state["c"] = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
        state["workspace"] = _workspace(find(m, n, k, bits, group))
    return state


def _gated(x, layer):
    op = torch.ops.awesome_fusion.bfaintb_gemm_prepacked if layer.prepacked else torch.ops.awesome_fusion.bfaintb_gemm
    return op(x, layer.qweight, layer.scales, layer.weight_bits, layer.group_size, None, None, 1)


def _prepare_block(g, case):
    h = case["k"]
    layers = [_quant_linear(g, n, k, case) for n, k in _block_shapes(case)]
    x = _normal(g, case["m"], h)

    def step():
        qkv = layers[0](x)
        y = layers[1](qkv[:, :h], residual=x)
        return {"qkv": qkv, "y": layers[3](_gated(y, layers[2]), residual=y)}

    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step()
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = step()
    return {"case": case, "layers": layers, "x": x, "graph": graph, "out": out}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return state["layer"](state["x"], residual=state["residual"])
    if kind == "gated":
        return _gated(state["x"], state["layer"])
    if kind == "abi":
        layer, c = state["layer"], state["c"]
        call = af.gemm_prepacked if case["packed"] else af.gemm
        call(c, state["x"], layer.qweight, layer.scales, case["m"], case["n"], case["k"], weight_bits=case["bits"],
             group_size=case["group"], workspace=state["workspace"], bias=layer.bias, residual=state["residual"])
        return c
    if kind == "block":
        state["graph"].replay()
        return state["out"]
    layer = top.QuantLinear.from_float(state["linear"], case["bits"], case["group"])
    if case["packed"]:
        layer.prepack()
    return {"qweight": layer.qweight, "scales": layer.scales}


def _gemm_work(m, n, k, case, out_n=None):
    groups = k // case["group"] if case["group"] else 1
    out_n = n if out_n is None else out_n
    return 2 * m * k + n * k * case["bits"] // 8 + 2 * groups * n + 2 * m * out_n, 2 * m * n * k


def work(case):
    m, n, k = case["m"], case["n"], case["k"]
    if case["kind"] == "load":
        groups = k // case["group"] if case["group"] else 1
        return {"bytes": 2 * n * k + n * k * case["bits"] // 8 + 2 * groups * n, "flops": 3 * n * k}
    if case["kind"] == "block":
        shapes = _block_shapes(case)
        parts = [_gemm_work(m, bn, bk, case, bn // 2 if i == 2 else bn) for i, (bn, bk) in enumerate(shapes)]
        parts.append((2 * m * k * 2, 0))  # the two residuals
    else:
        parts = [_gemm_work(m, n, k, case, n // 2 if case["kind"] == "gated" else n)]
        parts.append((2 * n * case["bias"] + 2 * m * n * case["residual"], 0))
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    if case["kind"] == "block":  # four bf16 roundings in a row
        return {"rel": 1e-2, "max": 5e-2}
    return {"rel": 4e-3, "max": 2e-2}  # one bf16 rounding of an fp32 sum: half a unit is 2^-9, two units 2^-6
