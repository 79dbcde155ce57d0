"""Timed cases of the EXL3 path: what a program that serves or converts EXL3 checkpoints
asks of this package, each through the public modules and functions.

Kinds (``"op"``):

* ``forward``: one call of ``EXL3Linear``, or of ``FusedEXL3Group.forward_all`` where
  ``outs`` lists several members that share an input. Launched eagerly, from one row (a
  decode step that nobody captured) over continuous batching to prefill chunks.
* ``decoder``: the linears of consecutive decoder layers (q+k+v, o, gate+up, down) at a
  decode or speculative-verify row count, captured once in a HIP graph and replayed, as
  a decoding loop does with its token step.
* ``moe``: one call of ``EXL3MoEBlock`` (router, routed experts, weighted sum), with or
  without a shared expert, from one token to a prefill chunk.
* ``encode``: ``quantize_inner_matrix_direct``, the converter's search and packing of one
  matrix.
* ``fold``: ``folded_linear_from_exl3``, an EXL3 layer turned into its plain fp16 linear.

Weights are random trellis words (every fill is a legal bitstream) with sign vectors
whose magnitude gives the public weights the scale of trained ones, 1/sqrt(in), so that
activations stay in the range that a model keeps them in; activations are fp16 N(0, 1).
"""

from __future__ import annotations

import math

import torch

from ponyexl3_amd import EXL3Layer, EXL3Linear, EXL3MoEBlock, EXL3SwitchGLU, FusedEXL3Group, clear_layer_caches
from ponyexl3_amd.native import folded_linear_from_exl3
from ponyexl3_amd.search import quantize_inner_matrix_direct

DEVICE = "cuda"
# standard deviation of the decoded codebook values
CODEBOOK_STD = 1.24


def _forward(name, rows, n_in, outs, k=4, cb=0, bias=False):
    return {"name": name, "op": "forward", "rows": rows, "in": n_in, "outs": outs, "k": k, "cb": cb, "bias": bias}


def _decoder(name, rows, hidden, q, kv, ffn, k=4, cb=0, layers=2):
    return {"name": name, "op": "decoder", "rows": rows, "hidden": hidden, "q": q, "kv": kv, "ffn": ffn, "k": k,
            "cb": cb, "layers": layers}


def _moe(name, tokens, dim, hidden, experts, top_k, shared, k=4, cb=0):
    return {"name": name, "op": "moe", "tokens": tokens, "dim": dim, "hidden": hidden, "experts": experts,
            "top_k": top_k, "shared": shared, "k": k, "cb": cb}


def listed():
    return [
        # the smallest linear of a 27B-class layer on its own: a k or v projection of one
        # token in a loop without graphs, all latency and launch cost
        _forward("k_proj 1 row", 1, 5120, "1024", bias=True),
        # single-stream decoding, the linears of two layers at the usual bit rate
        _decoder("decoder 1 row", 1, 5120, 8192, 1024, 17408),
        # speculative verification of a few drafted tokens, a higher bit rate
        _decoder("decoder 5 rows K6", 5, 5120, 8192, 1024, 17408, k=6, cb=1),
        # continuous batching: sixteen sequences decoding together
        _forward("gate_up 16 rows", 16, 5120, "17408,17408"),
        # a short prompt, ragged, on the attention projections
        _forward("qkv 77 rows", 77, 5120, "8192,1024,1024"),
        # the tail chunk of a prompt on the layer with the longest reduction
        _forward("down_proj 333 rows K5", 333, 17408, "5120", k=5, cb=1),
        # a full prefill chunk on the widest pair of linears
        _forward("gate_up 2048 rows", 2048, 5120, "17408,17408"),
        # routed experts of one decoded token
        _moe("moe 1 token", 1, 2048, 512, 256, 8, False),
        # a batch of sequences decoding together, with a shared expert
        _moe("moe 24 tokens", 24, 2048, 512, 256, 8, True),
        # a prefill chunk through the experts
        _moe("moe 1537 tokens", 1537, 2048, 512, 256, 8, True),
        # conversion of one projection-sized matrix
        {"name": "encode K3", "op": "encode", "in": 1024, "out": 1024, "k": 3, "cb": 1},
        # fp16 weight of a layer at load time
        {"name": "fold gate", "op": "fold", "in": 5120, "out": 17408, "k": 4, "cb": 0, "bias": False},
    ]


def _log_int(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + step - 1)))
    return max(lo, min(hi, int(v) // step * step))


def _codec(rng):
    # 4 bits is the common rate, 3INST and MCG the common codebooks
    return (4 if rng.random() < 0.3 else rng.randint(2, 8)), rng.choice((0, 0, 0, 1, 1, 1, 2))


def draw(rng):
    k, cb = _codec(rng)
    op = rng.choice(("forward", "forward", "forward", "forward", "decoder", "decoder", "moe", "moe", "moe", "encode",
                     "fold"))
    if op == "forward":
        rows = rng.choice((rng.randint(1, 8), rng.randint(9, 32), _log_int(rng, 33, 2048)))
        n_in = _log_int(rng, 1024, 17408, 128)
        shape = rng.randint(0, 2)
        if shape == 0:
            # a single linear; the widest of few rows are output heads
            outs = [_log_int(rng, 1024, 65536 if rows <= 32 else 17408, 128)]
        elif shape == 1:
            outs = [_log_int(rng, 1024, 17408, 128)] * 2
        else:
            kv = _log_int(rng, 256, 2048, 128)
            outs = [_log_int(rng, 1024, 8192, 128), kv, kv]
        # no larger than the widest pair of linears at a full chunk
        while n_in * sum(outs) > 5120 * 34816:
            n_in = n_in // 256 * 128
        case = _forward("", rows, n_in, ",".join(str(o) for o in outs), k, cb, len(outs) == 1 and rng.random() < 0.3)
    elif op == "decoder":
        hidden = _log_int(rng, 1024, 5120, 128)
        case = _decoder("", rng.choice((1, 1, rng.randint(2, 8))), hidden, hidden * rng.randint(6, 13) // 8 // 128 * 128,
                        rng.choice((256, 384, 512, 1024)), hidden * rng.randint(20, 27) // 8 // 128 * 128, k, cb,
                        rng.randint(1, 2))
    elif op == "moe":
        experts = rng.choice((32, 64, 128, 192, 256))
        case = _moe("", rng.choice((rng.randint(1, 8), _log_int(rng, 9, 1537))), _log_int(rng, 1024, 2048, 128),
                    _log_int(rng, 256, 768, 128), experts, rng.randint(4, 8), rng.random() < 0.5, k, cb)
        if case["tokens"] > 1 and case["dim"] * case["hidden"] > 2048 * 512:
            case["hidden"] = 512
    elif op == "encode":
        case = {"op": "encode", "in": _log_int(rng, 128, 1024, 128), "out": _log_int(rng, 128, 768, 128), "k": k,
                "cb": cb}
    else:
        case = {"op": "fold", "in": _log_int(rng, 512, 5120, 128), "out": _log_int(rng, 512, 17408, 128), "k": k,
                "cb": cb, "bias": rng.random() < 0.3}
    case.pop("name", None)
    return case


def _outs(case):
    return [int(o) for o in case["outs"].split(",")]


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _trellis(g, n_in, n_out, k):
    return torch.randint(-32768, 32768, (n_in // 16, n_out // 16, 16 * k), dtype=torch.int16, device=DEVICE, generator=g)


def _signs(g, *shape, scale=1.0):
    s = torch.randint(0, 2, shape, device=DEVICE, generator=g, dtype=torch.int8)
    return ((2 * s.to(torch.float32) - 1) * scale).to(torch.float16)


def _scale(n_in):
    return 1.0 / (CODEBOOK_STD * math.sqrt(n_in))


def _layer(g, key, n_in, n_out, k, cb, bias=False):
    """A layer record as a checkpoint reader fills it, on the host."""
    b = None
    if bias:
        b = (0.1 * torch.randn(n_out, device=DEVICE, generator=g)).half().cpu().numpy()
    return EXL3Layer(key=key, in_features=n_in, out_features=n_out, k=k,
                     trellis=_trellis(g, n_in, n_out, k).cpu().numpy().view("uint16"),
                     suh=_signs(g, n_in).cpu().numpy(), svh=_signs(g, n_out, scale=_scale(n_in)).cpu().numpy(), bias=b,
                     mcg=cb == 1, mul1=cb == 2)


def _linears(g, key, n_in, outs, k, cb, bias=False):
    layers = [_layer(g, f"{key}.{i}", n_in, o, k, cb, bias) for i, o in enumerate(outs)]
    return EXL3Linear(layers[0], DEVICE) if len(layers) == 1 else FusedEXL3Group(layers, DEVICE)


def _call(module, x):
    return module.forward_all(x) if isinstance(module, FusedEXL3Group) else module(x)


def _activations(g, *shape):
    return torch.randn(shape, device=DEVICE, generator=g).to(torch.float16)


def _prepare_decoder(case, g, seed):
    h, rows = case["hidden"], case["rows"]
    shapes = [(h, [case["q"], case["kv"], case["kv"]]), (case["q"], [h]), (h, [case["ffn"], case["ffn"]]),
              (case["ffn"], [h])]
    steps = []
    for layer in range(case["layers"]):
        for i, (n_in, outs) in enumerate(shapes):
            module = _linears(g, f"{seed}.{layer}.{i}", n_in, outs, case["k"], case["cb"])
            steps.append((module, _activations(g, rows, n_in)))

    def step():
        return [_call(module, x) for module, x in steps]

    # buffers of the capturing stream exist before the capture
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step()
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        outs = step()
    return {"op": "decoder", "graph": graph, "outs": outs, "steps": steps, "stream": stream}


def _prepare_moe(case, g):
    d, h, k = case["dim"], case["hidden"], case["k"]
    e = case["experts"] + int(case["shared"])
    switch = EXL3SwitchGLU(
        gu_trellis=_trellis(g, d, e * 2 * h, k), gu_suh=_signs(g, e, 2, d), gu_svh=_signs(g, e, 2 * h, scale=_scale(d)),
        dn_trellis=_trellis(g, h, e * d, k), dn_suh=_signs(g, e, h), dn_svh=_signs(g, e, d, scale=_scale(h)), k=k,
        cb=case["cb"])

    def gate(n):
        lin = torch.nn.Linear(d, n, bias=False, device="meta", dtype=torch.float16).to_empty(device=DEVICE)
        with torch.no_grad():  # router logits ~ N(0, 1)
            lin.weight.copy_(torch.randn((n, d), device=DEVICE, generator=g) / math.sqrt(d))
        return lin.requires_grad_(False)

    block = EXL3MoEBlock(gate(case["experts"]), gate(1) if case["shared"] else None, switch, case["top_k"])
    return {"op": "moe", "block": block, "x": _activations(g, case["tokens"], d)}


def prepare(case, seed):
    g = _generator(seed)
    op = case["op"]
    if op in ("forward", "decoder", "fold"):
        clear_layer_caches()  # device copies of layers that are gone
    if op == "forward":
        module = _linears(g, str(seed), case["in"], _outs(case), case["k"], case["cb"], case["bias"])
        return {"op": op, "module": module, "x": _activations(g, case["rows"], case["in"])}
    if op == "decoder":
        return _prepare_decoder(case, g, seed)
    if op == "moe":
        return _prepare_moe(case, g)
    if op == "encode":
        # regularised weights, which the converter scales to the codebook's spread
        return {"op": op, "k": case["k"], "cb": case["cb"],
                "inner": CODEBOOK_STD * torch.randn((case["in"], case["out"]), device=DEVICE, generator=g)}
    layer = _layer(g, str(seed), case["in"], case["out"], case["k"], case["cb"], case["bias"])
    EXL3Linear(layer, DEVICE)  # uploads the packed weights, as loading the model has done
    return {"op": op, "layer": layer}


@torch.no_grad()
def run(state):
    op = state["op"]
    if op == "forward":
        return _call(state["module"], state["x"])
    if op == "decoder":
        state["graph"].replay()
        return state["outs"]
    if op == "moe":
        return state["block"](state["x"])
    if op == "encode":
        packed, states, recon = quantize_inner_matrix_direct(state["inner"], k=state["k"], cb=state["cb"],
                                                             return_states=True)
        return {"packed": packed, "states": states, "recon": recon}
    linear = folded_linear_from_exl3(state["layer"])
    return {"weight": linear.weight} if linear.bias is None else {"weight": linear.weight, "bias": linear.bias}


def _linear_work(rows, n_in, outs, k, bias=False):
    n_out = sum(outs)
    return {"bytes": n_in * n_out * k / 8 + 2 * rows * (n_in + n_out) + 2 * (len(outs) * n_in + n_out * (1 + int(bias))),
            "flops": 2.0 * rows * n_in * n_out}


def work(case):
    op, k = case["op"], case["k"]
    if op == "forward":
        return _linear_work(case["rows"], case["in"], _outs(case), k, case["bias"])
    if op == "decoder":
        h, q, kv, f = case["hidden"], case["q"], case["kv"], case["ffn"]
        parts = [_linear_work(case["rows"], a, b, k) for a, b in ((h, [q, kv, kv]), (q, [h]), (h, [f, f]), (f, [h]))]
        return {m: case["layers"] * sum(p[m] for p in parts) for m in ("bytes", "flops")}
    if op == "moe":
        t, d, h, e, s = case["tokens"], case["dim"], case["hidden"], case["experts"], int(case["shared"])
        # experts that at least one of the tokens is expected to select
        used = e * (1.0 - (1.0 - case["top_k"] / e) ** t) + s
        weights = used * (3 * d * h * k / 8 + 2 * (2 * d + 3 * h + d)) + 2 * d * (e + s)
        return {"bytes": weights + 2 * 2 * t * d, "flops": 2.0 * t * ((case["top_k"] + s) * 3 * d * h + d * (e + s))}
    n = case["in"] * case["out"]
    if op == "encode":
        # two passes over 256 steps of a tile, 65 536 candidates each: difference, square,
        # sum, comparison; fp32 in, words, 16-bit states and fp32 values out
        return {"bytes": n * (4 + k / 8 + 2 + 4), "flops": n / 256 * 2 * 256 * 65536 * 4.0}
    # a Hadamard transform of 128 is seven additions per value and side
    return {"bytes": n * (k / 8 + 2) + 2 * (case["in"] + case["out"]), "flops": n * 2 * 7.0}


def tolerance(case):
    op = case["op"]
    if op == "encode":
        return "exact"  # ties go to the lowest state: one right answer
    if op == "moe":
        # three linears with fp16 between them, the gated product in the middle
        return {"rel": 2e-3, "max": 4e-2}
    # fp16 outputs, fp16 rotated activations, fp16 before the output transform
    return {"rel": 1e-3, "max": 2e-2}
