"""The workloads this package's speed is judged on: what an inference program has it do, through the public layers
and kernel factories, from one token's decode to a long prefill.

``listed()`` names twelve of them, ``draw(rng)`` gives more from the same ranges; ``prepare`` makes what the program
holds before the call (weights, scales, the layer or kernel object, for a decode loop the captured graph), ``run`` is
one pass.  Sizes are those of the benchmark configurations and tests (7B- and 70B-class projections, N = K = 8192, the
2880-wide MXFP4 matrices, 4096-wide W4A8) and generic odd ones between them.
"""

from __future__ import annotations

import torch

import tilelang_amd as tl
from tilelang_amd.bitlinear import BitLinear
from tilelang_amd.w4linear import W4A16Linear

# (N, K) of the projections of one decoder block, 7B class: q, k, v, o, gate, up, down
BLOCK_7B = ((4096, 4096),) * 4 + ((11008, 4096),) * 2 + ((4096, 11008),)


def _w4a16(name, rows, n, k, group=128, zeros=False):
    return {"name": name, "kind": "w4a16", "rows": rows, "n": n, "k": k, "group": group, "zeros": zeros, "block": False}


def _mxfp4(name, rows, n, k, bias=False):
    return {"name": name, "kind": "mxfp4", "rows": rows, "n": n, "k": k, "bias": bias}


def _bitlinear(name, rows, n, k, fragments=False):
    return {"name": name, "kind": "bitlinear", "rows": rows, "n": n, "k": k, "fragments": fragments, "block": False}


def listed():
    return [
        # one token through one layer, called from Python: the smallest call, latency and host work count
        _w4a16("w4a16 one row, one layer", 1, 4096, 4096),
        # one token through the seven projections of a 7B-class block, replayed from a graph: a serving loop's decode step
        {"name": "w4a16 decode block", "kind": "w4a16", "rows": 1, "n": 4096, "k": 4096, "group": 128, "zeros": False, "block": True},
        # sixteen sequences decoding together against a 70B-class feed-forward matrix, asymmetric quantisation
        _w4a16("w4a16 decode batch", 16, 28672, 8192, zeros=True),
        # one short prompt (or one chunk of a chunked prefill), odd length, 13B-class matrix, groups of 64
        _w4a16("w4a16 short prefill", 300, 13824, 5120, group=64, zeros=True),
        # a batch of prompts, 8B-class feed-forward down projection, symmetric quantisation
        _w4a16("w4a16 long prefill", 2048, 4096, 14336),
        # one token, MXFP4 weights whose rows are no multiple of a cache line (K = 2880), bias, called from Python
        _mxfp4("mxfp4 one row", 1, 5760, 2880, bias=True),
        # a full decode batch (or a prompt of a hundred tokens): too many rows for a streaming kernel, too few for big tiles
        _mxfp4("mxfp4 large batch", 96, 8192, 8192),
        # prefill at the benchmark's size, the largest case
        _mxfp4("mxfp4 prefill", 4096, 8192, 8192),
        # eight sequences decoding through a block of BitLinear layers (weights held in the operand order where a layer
        # can), replayed from a graph
        {"name": "bitlinear decode block", "kind": "bitlinear", "rows": 8, "n": 4096, "k": 4096, "fragments": True, "block": True},
        # a short prompt of odd length through a BitLinear layer
        _bitlinear("bitlinear short prefill", 200, 8192, 8192),
        # a long prompt through a BitLinear layer
        _bitlinear("bitlinear long prefill", 2048, 8192, 8192),
        # int8 activations on int4 weights, a ragged batch of prompts
        {"name": "w4a8 prefill", "kind": "w4a8", "rows": 1000, "n": 11008, "k": 4096},
    ]


def _log(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def draw(rng):
    kind = rng.choice(("w4a16", "w4a16", "mxfp4", "mxfp4", "bitlinear", "bitlinear", "w4a8"))
    # rows: one, a decode batch, a large batch or short prompt, a long prompt, in equal shares
    lo, hi = rng.choice(((1, 2), (2, 33), (33, 513), (513, 4097)))
    rows = min(int(_log(rng, lo, hi)), hi - 1)
    # most matrices have K % 256 == 0 (5120, 11008, 13824, ...); some only K % 128 == 0 (3200) or, MXFP4, K % 64 == 0 (2880)
    step = 256 if rng.random() < 0.75 else (64 if kind == "mxfp4" else 128)
    k = int(_log(rng, 2048, 14336)) // step * step
    n = int(_log(rng, 2048, 28672)) // 8 * 8
    # nothing costs more than the largest listed case (549.8 GFLOP in bf16)
    most = {"w4a16": 3.2e11, "mxfp4": 4.5e11, "bitlinear": 5e11, "w4a8": 5e11}[kind]
    if 2.0 * rows * n * k > most:
        rows = max(1, int(most / (2.0 * n * k)))
    if kind == "w4a8":
        return {"kind": kind, "rows": rows, "n": n, "k": k}
    if kind == "mxfp4":
        return {"kind": kind, "rows": rows, "n": n, "k": k, "bias": rng.random() < 0.25}
    # decode batches come both ways: one layer from Python, a block of layers from a graph
    block = rows <= 32 and rng.random() < 0.5
    if kind == "bitlinear":
        return {"kind": kind, "rows": rows, "n": n, "k": k, "fragments": rng.random() < 0.5, "block": block}
    # the layer's groups divide K: 128 always does, 64 always does
    return {"kind": kind, "rows": rows, "n": n, "k": k, "group": 64 if rng.random() < 0.25 else 128, "zeros": rng.random() < 0.5,
            "block": block}


def _shapes(case):
    """(N, K) of every layer of the case: a block is q, k, v, o on [k, k], gate and up on [n, k], down on [k, n']
    (the feed-forward width rounded up to what a layer's K allows), or the 7B-class block where n = k = 4096."""
    n, k = case["n"], case["k"]
    if not case.get("block"):
        return ((n, k),)
    if (n, k) == (4096, 4096):
        return BLOCK_7B
    wide = (n + 255) // 256 * 256
    return ((k, k),) * 4 + ((wide, k),) * 2 + ((k, wide),)


class _Inputs:
    """Random inputs on the GPU, from the seed alone."""

    def __init__(self, seed):
        self.dev = torch.device("cuda")
        self.gen = torch.Generator(device=self.dev)
        self.gen.manual_seed(seed)

    def normal(self, *shape, dtype):
        return torch.randn(shape, dtype=torch.float32, device=self.dev, generator=self.gen).to(dtype)

    def uniform(self, lo, hi, *shape):
        return (torch.rand(shape, device=self.dev, generator=self.gen) * (hi - lo) + lo).half()

    def ints(self, lo, hi, *shape, dtype):
        """lo .. hi inclusive"""
        return torch.randint(lo, hi + 1, shape, device=self.dev, generator=self.gen, dtype=dtype)

    def packed(self, *shape):
        """Bytes of packed codes, every code as likely as the next."""
        return self.ints(-128, 127, *shape, dtype=torch.int8)

    def ternary(self, n, k):
        """Codes w + 2 of w in {-1, 0, 1}, a third each, four per byte (in whatever order of k the layer's words have)."""
        c = self.ints(1, 3, n, k // 4, 4, dtype=torch.uint8)
        return (c[..., 0] | (c[..., 1] << 2) | (c[..., 2] << 4) | (c[..., 3] << 6)).view(torch.int8)


def _captured(forward):
    """What a decode loop keeps: one step, warmed up and captured; its outputs are the graph's own buffers."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        forward()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outputs = forward()
    return graph, outputs


def _drawn(case, make):
    """The inputs of a kernel case, in the order that its call takes them."""
    rows, n, k = case["rows"], case["n"], case["k"]
    if case["kind"] == "w4a8":
        return make.ints(-128, 127, rows, k, dtype=torch.int8), make.packed(n, k // 2).view(torch.uint8)
    weight = make.packed(n, k // 2).view(torch.uint8)
    scale = make.ints(127 - 8, 127, n, k // 32, dtype=torch.uint8)
    bias = make.normal(rows, n, dtype=torch.bfloat16)
    return make.normal(rows, k, dtype=torch.bfloat16), weight, scale, bias


def _drawn_layers(case, make, seed):
    """For every layer of a case of layers: the tensors that it holds, and its activations."""
    for n, k in _shapes(case):
        if case["kind"] == "w4a16":
            held = {"qweight": make.packed(n, k // 2), "scales": make.uniform(0.002, 0.01, n, k // case["group"])}
            if case["zeros"]:
                held["zeros"] = make.ints(6, 10, n, k // case["group"], dtype=torch.int8).half()
        else:
            held = {"qweight": make.ternary(n, k), "sw": 1.0 + (seed % 7) / 4}
        yield n, k, held, make.normal(case["rows"], k, dtype=torch.float16)


def prepare(case, seed):
    kind, rows = case["kind"], case["rows"]
    make = _Inputs(seed)
    if kind in ("mxfp4", "w4a8"):
        n, k = case["n"], case["k"]
        if kind == "w4a8":
            kernel = tl.matmul_int8xint4(rows, n, k)
        else:
            kernel = tl.matmul_bf16_mxfp4(rows, n, k, with_bias=case["bias"], weight_format="e2m1", scale_bias=127)
        return {"kernel": kernel, "args": _drawn(case, make)}

    layers, inputs = [], []
    for n, k, held, x in _drawn_layers(case, make, seed):
        if kind == "w4a16":
            layer = W4A16Linear(k, n, group_size=case["group"], with_zeros=case["zeros"]).to(make.dev)
            layer.load_state_dict(held)
        else:
            layer = BitLinear(k, n, prefill_fragments=case["fragments"]).to(make.dev)
            layer.load_packed_weight(held["qweight"], held["sw"])
        layers.append(layer)
        inputs.append(x)
    state = {"layers": layers, "inputs": inputs}
    if case["block"]:
        with torch.no_grad():
            state["graph"], state["outputs"] = _captured(lambda: [layer(x) for layer, x in zip(layers, inputs)])
    return state


def run(state):
    if "kernel" in state:
        return state["kernel"](*state["args"])
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    with torch.no_grad():
        return state["layers"][0](state["inputs"][0])


def work(case):
    kind, rows = case["kind"], case["rows"]
    moved = done = 0
    for n, k in _shapes(case):
        done += 2 * rows * n * k
        if kind == "w4a16":
            moved += n * k // 2 + 2 * n * (k // case["group"]) * (2 if case["zeros"] else 1) + 2 * rows * (k + n)
        elif kind == "mxfp4":
            moved += n * k // 2 + n * (k // 32) + 2 * rows * k + 2 * rows * n * (2 if case["bias"] else 1)
        elif kind == "bitlinear":  # fp16 activations in, fp16 out; the int8 copy between the two kernels need not reach memory
            moved += n * k // 4 + 2 * rows * (k + n)
        else:
            moved += n * k // 2 + rows * k + 4 * rows * n
    return {"bytes": moved, "flops": done}


def tolerance(case):
    """About four times the distance from the same computation in float64 (measured over the listed and ten drawn cases)."""
    return {
        # the fp16 result's rounding alone is 2.1e-4 (largest 4.9e-4); kernels that round every weight to fp16, or the product
        # of zero point and scale, come to 2.7e-4 ... 4.4e-4 (largest 1.8e-3)
        "w4a16": {"rel": 1.8e-3, "max": 7e-3},
        # the bf16 result's rounding: 1.67e-3, largest 3.9e-3
        "mxfp4": {"rel": 6.5e-3, "max": 1.6e-2},
        # the sums are exact integers: the fp16 result's rounding
        "bitlinear": {"rel": 8e-4, "max": 2e-3},
        "w4a8": "exact",
    }[case["kind"]]


def _nibbles(packed):
    """Codes 0 .. 15 of packed bytes, the even column in the low nibble."""
    b = packed.view(torch.uint8)
    return torch.stack((b & 15, b >> 4), dim=-1).reshape(b.shape[0], -1)


def _ternary_codes(packed):
    """Codes of words whose element e lies at bit 8 * (e % 4) + 2 * (e // 4)."""
    b = packed.view(torch.uint8).reshape(packed.shape[0], -1, 1, 4)
    shift = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=b.device).view(1, 1, 4, 1)
    return ((b >> shift) & 3).reshape(packed.shape[0], -1)


def exact(case, seed):
    """The result in 64 bits.  A BitLinear layer's activations are whole numbers that 32-bit arithmetic defines (127 over
    the row's largest magnitude, to the nearest): they are taken so, and all after them in 64 bits."""
    kind = case["kind"]
    make = _Inputs(seed)
    if kind == "w4a8":
        a, packed = _drawn(case, make)
        codes = _nibbles(packed).to(torch.int16)
        return (torch.where(codes > 7, codes - 16, codes).double() @ a.double().t()).to(torch.int32)
    if kind == "mxfp4":
        a, packed, scale, bias = _drawn(case, make)
        values = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], dtype=torch.float64, device=make.dev)
        weight = torch.cat((values, -values))[_nibbles(packed).int()]
        weight = weight * torch.exp2(scale.double() - 127).repeat_interleave(32, dim=1)
        out = a.double() @ weight.t()
        return out + bias.double() if case["bias"] else out

    outputs = []
    for _, k, held, x in _drawn_layers(case, make, seed):
        if kind == "w4a16":
            codes = _nibbles(held["qweight"]).double()
            zeros = held["zeros"].double().repeat_interleave(case["group"], dim=1) if case["zeros"] else 8.0
            outputs.append(x.double() @ ((codes - zeros) * held["scales"].double().repeat_interleave(case["group"], dim=1)).t())
        else:
            s = 127 / x.float().abs().amax(dim=1, keepdim=True).clamp(min=1e-5)
            whole = (x.float() * s).round().clamp(-128, 127).double()
            outputs.append(whole @ (_ternary_codes(held["qweight"]).double() - 2).t() / s.double() / held["sw"])
    return outputs if case["block"] else outputs[0]
