"""What this framework is timed on: the quantized layers of a decode step, a tree-verify step and a
prefill, each through the entry point that a program calls.

A pass runs `layers` layers of one kind one after another, each on weights of its own, as a forward
does: a forward's next layer is never in the caches, so a case with small weights holds several.
Sizes are those of the target model of tests and benchmark (hidden 5120, MLP 17408, fused gate+up
34816, vocabulary 151936), at the row counts of decode (1-4), a tree-verify batch (5-64), a short
prompt tail (65-512) and a prefill chunk (up to 4096).

A case's `op`:
  norm          add_rms_norm: the residual add and RMS norm between two projections
  linear        an installed QuantizedLinear, y = x @ dequant(w).T (eligible shapes run the packed
                kernels; other shapes and formats the dequantization and a bf16 product)
  gate_up       gate_up_silu: the MLP's fused gate+up projection with SiLU * mul
  norm_gate_up  add_rms_norm_gate_up: that norm folded into the gate+up projection
  tail          stack_tail captured in a HIP graph (GraphedTail): the MLP half of a forward
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mlx-tree-spec_amd"))

from mlx_tree_spec_amd import (  # noqa: E402
    GraphedTail, MLPLayer, QuantizedLinear, QuantizedMLP, add_rms_norm, add_rms_norm_gate_up, gate_up_silu, install)

EPS = 1e-6
LARGEST_MNK = 4096 * 5120 * 17408  # the largest listed case
LARGEST_NK = 151936 * 5120         # the largest weight matrix


def _case(name, op, m, k=0, n=0, layers=1, bits=4, group=64):
    return {"name": name, "op": op, "m": m, "k": k, "n": n, "layers": layers, "bits": bits, "group": group}


def listed():
    return [
        # The smallest call: a decode step's residual add + norm over 3 requests.
        _case("norm 3x5120", "norm", 3, 5120),
        # Decode, one request: the norm folded into the fused gate+up projection.
        _case("decode norm+gate_up 1x5120-34816", "norm_gate_up", 1, 5120, 34816, layers=2),
        # Decode, 4 batched requests: the MLP's down projection.
        _case("decode down 4x17408-5120", "linear", 4, 17408, 5120, layers=4),
        # Decode as a serving loop runs it: the MLP half of 4 layers replayed as one graph, 2 requests.
        _case("decode tail graph 2 rows", "tail", 2, 5120, 34816, layers=4),
        # One request's tree verify (16 nodes): an attention-sized square projection.
        _case("verify 16x5120-5120", "linear", 16, 5120, 5120, layers=8),
        # A ragged tree (13 nodes): the fused gate+up.
        _case("verify gate_up 13x5120-34816", "gate_up", 13, 5120, 34816, layers=2),
        # Batched tree verify (4 requests x 16 nodes): the down projection.
        _case("verify down 64x17408-5120", "linear", 64, 17408, 5120, layers=4),
        # The vocabulary head at verify: the largest weight stream of a step.
        _case("verify head 32x5120-151936", "linear", 32, 5120, 151936),
        # A short prompt tail of odd length: the up projection.
        _case("prompt tail up 203x5120-17408", "linear", 203, 5120, 17408, layers=2),
        # A prompt chunk that is not a multiple of the tiles: the down projection.
        _case("prompt down 1000x17408-5120", "linear", 1000, 17408, 5120),
        # Chunked prefill, the compute-bound end: the up projection over 4096 tokens.
        _case("prefill up 4096x5120-17408", "linear", 4096, 5120, 17408),
        # A layer that the packed kernels do not take: 8-bit codes in groups of 32, ragged columns.
        _case("8-bit 24x2560-4100", "linear", 24, 2560, 4100, layers=4, bits=8, group=32),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    op = rng.choice(["norm", "linear", "linear", "linear", "linear", "linear", "gate_up", "norm_gate_up", "tail", "format"])
    k = 128 * round(_log_uniform(rng, 1024, 17408) / 128)
    if op == "norm":
        return _draw("norm", round(_log_uniform(rng, 1, 4096)), 8 * round(_log_uniform(rng, 1024, 8192) / 8), 0)
    if op == "format":  # the general path
        bits, group = rng.choice([(2, 64), (4, 32), (4, 64), (4, 128), (8, 32), (8, 64)])
        m, n = round(_log_uniform(rng, 1, 512)), round(_log_uniform(rng, 512, 8192)) | 1
        return _draw("linear", m, min(k, 8192), n, bits=bits, group=group)
    # Decode, verify, prompt tail and prefill as often as each other.
    lo, hi = rng.choice([(1, 4), (5, 16), (17, 64), (65, 512), (513, 4096)])
    m = round(_log_uniform(rng, lo, hi))
    if op == "tail":  # up to 64 rows: decode and verify steps
        return _draw("tail", min(m, 64), 128 * round(_log_uniform(rng, 1024, 5120) / 128),
                     256 * round(_log_uniform(rng, 4096, 34816) / 256), layers=2)
    if op in ("gate_up", "norm_gate_up"):
        n = 64 * round(_log_uniform(rng, 2048, 34816) / 64)
    else:  # a vocabulary head now and then, else a layer's projection
        n = 32 * round(_log_uniform(rng, 512, 17408) / 32) if rng.random() < 0.8 else 32 * round(_log_uniform(rng, 32768, 151936) / 32)
    k = min(k, 128 * (LARGEST_NK // (n * 128)))
    m = max(1, min(m, LARGEST_MNK // (n * k)))
    return _draw(op, m, k, n)


def _draw(op, m, k, n, layers=0, bits=4, group=64):
    # Layers enough for about 100 MB of weights, at most 8, as in the listed cases.
    if not layers:
        layers = 1 if op == "norm" or m > 512 else max(1, min(8, round(1e8 / max(1, n * k * bits / 8))))
    return {"op": op, "m": m, "k": k, "n": n, "layers": layers, "bits": bits, "group": group}


# Inputs: activations after a norm are about N(0, 1) (0.5 in front of a down projection); codes are
# uniform; scales and biases as affine quantization of trained weights gives them (codes centred on
# zero, so the bias is about -mid * scale).

def _randn(gen, *shape, std=1.0):
    return (torch.randn(*shape, generator=gen, device="cuda") * std).to(torch.bfloat16)


def _weights(gen, n, k, bits, group):
    w = torch.randint(-2**31, 2**31, (n, k * bits // 32), generator=gen, device="cuda", dtype=torch.int64).to(torch.int32)
    s = (torch.randn(n, k // group, generator=gen, device="cuda").abs() * 0.004 + 1e-4) * 2.0 ** (4 - bits)
    s = s.to(torch.bfloat16)
    b = -(2.0 ** (bits - 1)) * s.float() + torch.randn(n, k // group, generator=gen, device="cuda") * 1e-3
    return w, s, b.to(torch.bfloat16)


def _norm(gen, dim):
    norm = torch.nn.RMSNorm(dim, eps=EPS, device="cuda", dtype=torch.bfloat16)
    norm.weight.requires_grad_(False)
    norm.weight.copy_(1.0 + 0.1 * torch.randn(dim, generator=gen, device="cuda"))
    return norm


def _raw(case, seed):
    """The case's inputs, from the seed alone: a list of per-layer dicts."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    op, m, k, n, bits, group = (case[f] for f in ("op", "m", "k", "n", "bits", "group"))
    out = []
    for _ in range(case["layers"]):
        d = {"x": _randn(gen, m, k, std=0.5 if k > 6144 else 1.0)}
        if op in ("norm", "norm_gate_up", "tail"):
            d["r"] = _randn(gen, m, k)
            d["norm"] = _norm(gen, k)
        if op != "norm":
            d["w"] = _weights(gen, n, k, bits, group)
        if op == "tail":
            d["down"] = _weights(gen, k, n // 2, bits, group)
            d["next"] = _norm(gen, k)
        out.append(d)
    return out


def _mlp(d, k, n):
    w, s, b = d["w"]
    half = n // 2
    gate, up = (QuantizedLinear.from_quantized(w[i:i + half], s[i:i + half], b[i:i + half]) for i in (0, half))
    if "down" not in d:  # the projection alone is run: any down projection of the right shape
        down = QuantizedLinear(half, k, device="cuda")
    else:
        down = QuantizedLinear.from_quantized(*d["down"])
    return QuantizedMLP(gate, up, down)


def prepare(case, seed):
    op, m, k, n = (case[f] for f in ("op", "m", "k", "n"))
    layers = _raw(case, seed)
    if op == "linear":
        mods = [QuantizedLinear.from_quantized(*d["w"], group_size=case["group"], bits=case["bits"]) for d in layers]
        install(torch.nn.ModuleList(mods), verbose=False)
        return {"op": op, "layers": [(mod, d["x"]) for mod, d in zip(mods, layers)]}
    if op == "tail":
        stack = [MLPLayer(d["norm"], _mlp(d, k, n)) for d in layers]
        install(torch.nn.ModuleList(stack), verbose=False)
        with torch.no_grad():
            graphed = GraphedTail(stack, layers[-1]["next"], m, k, "cuda")
        return {"op": op, "graph": graphed, "h": layers[0]["x"], "r": [d["r"] for d in layers]}
    if op == "norm_gate_up":
        return {"op": op, "layers": [(d["x"], d["r"], d["norm"], _mlp(d, k, n)) for d in layers]}
    return {"op": op, "layers": layers}


def run(state):
    op = state["op"]
    with torch.no_grad():
        if op == "linear":
            return [mod(x) for mod, x in state["layers"]]
        if op == "tail":
            return state["graph"](state["h"], state["r"])
        if op == "norm_gate_up":
            return [add_rms_norm_gate_up(x, r, norm, mlp) for x, r, norm, mlp in state["layers"]]
        if op == "gate_up":
            return [gate_up_silu(d["x"], *d["w"]) for d in state["layers"]]
        return [add_rms_norm(d["x"], d["r"], d["norm"]) for d in state["layers"]]


def _weight_bytes(n, k, bits, group):
    return n * k * bits // 8 + 4 * n * (k // group)


def work(case):
    op, m, k, n, layers, bits, group = (case[f] for f in ("op", "m", "k", "n", "layers", "bits", "group"))
    mk = 2 * m * k
    if op == "norm":
        return {"bytes": layers * (4 * mk + 2 * k), "flops": 0}
    flops = 2 * m * n * k
    nbytes = _weight_bytes(n, k, bits, group)
    if op == "linear":
        nbytes += mk + 2 * m * n
    elif op == "gate_up":
        nbytes += mk + m * n
    elif op == "norm_gate_up":
        nbytes += 4 * mk + 2 * k + m * n
    else:  # tail: the residual stream stays with the graph; each layer reads its r
        nbytes += _weight_bytes(k, n // 2, bits, group) + mk + 4 * k
        flops += 2 * m * k * (n // 2)
    extra = 3 * mk if op == "tail" else 0  # h in, h and x out
    return {"bytes": layers * nbytes + extra, "flops": layers * flops}


def tolerance(case):
    # The paths against 64 bits: 1.7e-3 (one bf16 rounding of the result, the weights' own rounding
    # being part of the format), 3e-3 behind a norm, 3.8e-3 with the SiLU * mul's three roundings
    # and 5.6e-3 with both. `max`: a result next to a rounding boundary differs by one bf16 step,
    # 2^-7 of it, and more where products cancel.
    op = case["op"]
    if op == "norm":
        return {"rel": 5e-3, "max": 0.016}
    if op == "linear":
        return {"rel": 6e-3, "max": 0.03}
    if op == "tail":
        return {"rel": 1.2e-2, "max": 0.1}
    return {"rel": 1e-2, "max": 0.06}


def _exact_matmul(x, weights, bits, group):
    """x (fp64) @ dequant(w).T in fp64; a dequantized weight is bf16(fp32(s) * q + fp32(b))."""
    w, s, b = weights
    n = w.shape[0]
    per = 32 // bits
    shifts = torch.arange(per, device=w.device, dtype=torch.int32) * bits
    out = []
    step = max(1, (1 << 28) // (w.shape[1] * per))
    for i in range(0, n, step):
        q = (w[i:i + step, :, None] >> shifts) & (2**bits - 1)
        q = q.reshape(q.shape[0], -1, group).double()
        v = (s[i:i + step, :, None].double() * q + b[i:i + step, :, None].double()).float().to(torch.bfloat16)
        out.append(x @ v.double().reshape(q.shape[0], -1).T.contiguous())
    return torch.cat(out, 1)


def _exact_norm(x, r, norm):
    h = x.double() + r.double()
    n = h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * norm.weight.double()
    return h, n


def _exact_silu_mul(t):
    g, u = t.chunk(2, 1)
    return torch.nn.functional.silu(g) * u


def exact(case, seed):
    op, bits, group = case["op"], case["bits"], case["group"]
    layers = _raw(case, seed)
    with torch.no_grad():
        if op == "norm":
            return [_exact_norm(d["x"], d["r"], d["norm"]) for d in layers]
        if op == "linear":
            return [_exact_matmul(d["x"].double(), d["w"], bits, group) for d in layers]
        if op == "gate_up":
            return [_exact_silu_mul(_exact_matmul(d["x"].double(), d["w"], bits, group)) for d in layers]
        if op == "norm_gate_up":
            out = []
            for d in layers:
                h, n = _exact_norm(d["x"], d["r"], d["norm"])
                out.append((h, n, _exact_silu_mul(_exact_matmul(n, d["w"], bits, group))))
            return out
        h, x = layers[0]["x"].double(), None
        for i, d in enumerate(layers):
            h, x = _exact_norm(h, d["r"], d["norm"])
            t = _exact_matmul(_exact_silu_mul(_exact_matmul(x, d["w"], bits, group)), d["down"], bits, group)
            h, x = _exact_norm(h, t, layers[i + 1]["norm"] if i + 1 < len(layers) else d["next"])
        return h, x
