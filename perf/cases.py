"""The workloads this package is timed on: what a decoding engine asks of it, from one token to a long prompt.

Three families, each through the entry points an engine calls:

    glu      blocks.BlockSwitchGLU, a layer's routed experts (gate, up, SwiGLU, down) at 1 to 8192 tokens
    linear   dense.BlockLinear, a projection or output layer kept as the file's blocks, at 1 to 2048 tokens
    moe      fused.RoutedMoE, the whole MoE block (router, choice, routed and shared experts, combine)

Shapes are those of the benchmark (256 experts top-8, 1536 x 4096; attention 4096 x 4096, lm_head 151936 x 4096) and
the second model shape of the tests and baseline (512 experts top-10, 640 x 2560). Blocks are random bytes with
|N(0, 1)| * 0.01 scales and routing is Zipf(1.1), as the benchmark draws them.

A decode step (`layers` > 0) is captured once as a HIP graph over that many distinct layers, enough that the weights
do not stay in the 256 MB cache from one pass to the next, and replayed, as an engine's decode loop does; each layer
has its own token. Longer calls are made eagerly.
"""

import math

import numpy as np
import torch

from strata_mlx_amd import blocks as B
from strata_mlx_amd import dense as D
from strata_mlx_amd import fused as Fu
from strata_mlx_amd import synth

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
# experts, top-k, ffn width, hidden width
SHAPES = {"a": (256, 8, 1536, 4096), "b": (512, 10, 640, 2560)}
BLOCK = {"IQ4_NL": (32, 18), "IQ3_S": (256, 110), "IQ3_XXS": (256, 98), "Q2_0": (64, 18), "Q8_0": (32, 34),
         "Q4_K": (256, 144), "Q6_K": (256, 210)}
# rough root mean square of a random block's weights: the activations are scaled so that gate and up come out near 1
WEIGHT_RMS = {"IQ4_NL": 0.7, "IQ3_S": 1.4, "IQ3_XXS": 1.8, "Q2_0": 0.012, "Q8_0": 0.74, "Q4_K": 3.3, "Q6_K": 13.5}


def listed():
    return [
        # one decode token through four whole MoE blocks: the step whose latency an interactive user waits for
        {"name": "moe_token", "family": "moe", "tokens": 1, "layers": 4},
        # a bfloat16 model's decode token through its routed experts
        {"name": "glu_token_bf16", "family": "glu", "shape": "a", "gate": "IQ3_S", "down": "IQ3_S", "dtype": "bf16",
         "tokens": 1, "layers": 5},
        # a speculative window: the last token and four drafts verified together
        {"name": "glu_verify5_q2", "family": "glu", "shape": "a", "gate": "Q2_0", "down": "Q2_0", "dtype": "f16",
         "tokens": 5, "layers": 3},
        # a server's batch: 48 requests decoding together
        {"name": "glu_batch48_bf16", "family": "glu", "shape": "a", "gate": "IQ3_S", "down": "IQ3_S", "dtype": "bf16",
         "tokens": 48, "layers": 0},
        # an ordinary prompt chunk
        {"name": "glu_prompt512_bf16", "family": "glu", "shape": "a", "gate": "IQ3_XXS", "down": "IQ3_XXS",
         "dtype": "bf16", "tokens": 512, "layers": 0},
        # the largest: a long prompt in one call
        {"name": "glu_prompt8192_bf16", "family": "glu", "shape": "a", "gate": "IQ3_S", "down": "IQ3_S",
         "dtype": "bf16", "tokens": 8192, "layers": 0},
        # a prompt of an odd length through the many small experts of the second shape, down in another type
        {"name": "glu_prompt1022_mixed", "family": "glu", "shape": "b", "gate": "IQ3_XXS", "down": "IQ4_NL",
         "dtype": "f16", "tokens": 1022, "layers": 0},
        # a prompt through a model of the common 4-bit mix: gate and up in Q4_K, down in Q6_K
        {"name": "glu_prompt384_q4k_q6k", "family": "glu", "shape": "a", "gate": "Q4_K", "down": "Q6_K",
         "dtype": "bf16", "tokens": 384, "layers": 0},
        # the q/k/v projections of one decode token, eight layers of a step
        {"name": "linear_qkv_token", "family": "linear", "kind": "Q6_K", "rows": 12288, "cols": 4096, "dtype": "f16",
         "tokens": 1, "layers": 8},
        # the output layer over a speculative window
        {"name": "linear_head_verify5", "family": "linear", "kind": "Q6_K", "rows": 151936, "cols": 4096,
         "dtype": "f16", "tokens": 5, "layers": 0},
        # a projection at a server's batch or a short prompt, a ragged number of tokens
        {"name": "linear_batch77_bf16", "family": "linear", "kind": "Q4_K", "rows": 4096, "cols": 4096,
         "dtype": "bf16", "tokens": 77, "layers": 0},
        # the q/k/v projections of a prefill chunk
        {"name": "linear_prefill2048_bf16", "family": "linear", "kind": "Q6_K", "rows": 12288, "cols": 4096,
         "dtype": "bf16", "tokens": 2048, "layers": 0},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    u = rng.random()
    if u < 0.1:
        return {"family": "moe", "tokens": _log(rng, 1, 16), "layers": 0}
    if u < 0.6:
        shape = rng.choice(["a", "a", "b"])
        if shape == "a":
            gate, down = rng.choice([("IQ3_S", "IQ3_S"), ("IQ3_XXS", "IQ3_XXS"), ("Q2_0", "Q2_0"), ("Q4_K", "Q6_K"),
                                     ("Q4_K", "Q4_K")])
        else:
            gate, down = rng.choice([("IQ3_XXS", "IQ4_NL"), ("Q2_0", "Q2_0"), ("IQ3_S", "IQ4_NL")])
        # the 4-bit mix through the routed kernels costs several times the codebook types' time a token
        most = 640 if gate == "Q4_K" else 8192 if shape == "a" else 4096
        tokens = _log(rng, 1, most)
        return {"family": "glu", "shape": shape, "gate": gate, "down": down, "dtype": rng.choice(["f16", "bf16"]),
                "tokens": tokens, "layers": 2 if tokens <= 8 else 0}
    kind = rng.choice(["Q4_K", "Q6_K", "Q8_0"])
    cols = rng.choice([1536, 2560, 4096])
    tokens = _log(rng, 1, 2048)
    rows = _log(rng, 1024, 151936 if tokens <= 64 else 16384)
    if rng.random() < 0.7:
        rows = rows // 64 * 64
    dtype = rng.choice(["f16", "bf16"]) if tokens > 8 or rng.random() < 0.8 else "f32"
    return {"family": "linear", "kind": kind, "rows": rows, "cols": cols, "dtype": dtype, "tokens": tokens,
            "layers": 4 if tokens <= 8 else 0}


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _parts(case, seed):
    """A case's layers as plain tensors: for each, its blocks, tokens and routing."""
    g = _generator(seed)
    dev = torch.device("cuda")
    rng = np.random.default_rng(seed)
    tokens, parts = case["tokens"], []
    for _ in range(max(1, case["layers"])):
        if case["family"] == "linear":
            parts.append({"w": synth.random_stack(case["kind"], case["rows"] * case["cols"], dev, g),
                          "x": (torch.randn((tokens, case["cols"]), device=dev, generator=g) / 8).to(DTYPES[case["dtype"]])})
            continue
        moe = case["family"] == "moe"
        experts, k, ffn, hidden = SHAPES["a" if moe else case["shape"]]
        gate, down = ("IQ3_S", "IQ3_S") if moe else (case["gate"], case["down"])
        dtype = torch.float16 if moe else DTYPES[case["dtype"]]
        p = {"gate": synth.random_stack(gate, experts * ffn * hidden, dev, g),
             "up": synth.random_stack(gate, experts * ffn * hidden, dev, g),
             "down": synth.random_stack(down, experts * hidden * ffn, dev, g),
             "x": (torch.randn((tokens, hidden), device=dev, generator=g) / (math.sqrt(hidden) * WEIGHT_RMS[gate])).to(dtype)}
        if moe:
            p["router"] = torch.randn((experts, hidden), device=dev, generator=g).half()
            p["shared_expert_gate"] = torch.randn((1, hidden), device=dev, generator=g).half()
            for name in ("shared_gate", "shared_up", "shared_down"):
                p[name] = synth.random_stack("Q4_K", ffn * hidden, dev, g)
        else:
            p["idx"] = torch.from_numpy(synth.zipf_routing(tokens, experts, k, rng)[0]).to(torch.int32).to(dev)
        parts.append(p)
    return parts


def _layer(case, p):
    """The object an engine keeps for a layer, and its call on the layer's input."""
    if case["family"] == "linear":
        lin = D.BlockLinear(p["w"], case["kind"], (case["rows"], case["cols"]))
        return lambda: lin(p["x"])
    moe = case["family"] == "moe"
    experts, k, ffn, hidden = SHAPES["a" if moe else case["shape"]]
    gate, down = ("IQ3_S", "IQ3_S") if moe else (case["gate"], case["down"])
    glu = B.BlockSwitchGLU(B.BlockSwitchLinear(p["gate"], gate, (experts, ffn, hidden)),
                           B.BlockSwitchLinear(p["up"], gate, (experts, ffn, hidden)),
                           B.BlockSwitchLinear(p["down"], down, (experts, hidden, ffn)))
    if not moe:
        return lambda: glu(p["x"], p["idx"])
    block = Fu.RoutedMoE(Fu.WindowLinear(p["router"]), glu, D.BlockLinear(p["shared_gate"], "Q4_K", (ffn, hidden)),
                         D.BlockLinear(p["shared_up"], "Q4_K", (ffn, hidden)),
                         D.BlockLinear(p["shared_down"], "Q4_K", (hidden, ffn)),
                         Fu.WindowLinear(p["shared_expert_gate"]), k)
    return lambda: block(p["x"])


def prepare(case, seed):
    calls = [_layer(case, p) for p in _parts(case, seed)]
    if not case["layers"]:
        return {"call": calls[0]}
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # one pass first: the library's and the allocator's lazy state
        for call in calls:
            call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = [call() for call in calls]
    return {"graph": graph, "outs": outs, "calls": calls}


def run(state):
    if "call" in state:
        return state["call"]()
    state["graph"].replay()
    return state["outs"]


def _row_bytes(kind, cols):
    per, size = BLOCK[kind]
    return cols // per * size


def work(case):
    n, t = max(1, case["layers"]), case["tokens"]
    if case["family"] == "linear":
        e = 4 if case["dtype"] == "f32" else 2
        rows, cols = case["rows"], case["cols"]
        return {"bytes": n * (rows * _row_bytes(case["kind"], cols) + t * (rows + cols) * e),
                "flops": n * 2.0 * t * rows * cols}
    moe = case["family"] == "moe"
    experts, k, ffn, hidden = SHAPES["a" if moe else case["shape"]]
    gate, down = ("IQ3_S", "IQ3_S") if moe else (case["gate"], case["down"])
    expert = 2 * ffn * _row_bytes(gate, hidden) + hidden * _row_bytes(down, ffn)
    if moe:  # its routing is the router's own: near enough uniform
        used = experts * (1 - (1 - k / experts) ** t)
        extra = 2 * ffn * _row_bytes("Q4_K", hidden) + hidden * _row_bytes("Q4_K", ffn) + (experts + 1) * hidden * 2
        return {"bytes": n * (used * expert + extra + t * 2 * hidden * 2),
                "flops": n * 2.0 * t * ((k + 1) * 3 * ffn * hidden + (experts + 1) * hidden)}
    # the distinct experts that a routing of this size names
    used = len(np.unique(synth.zipf_routing(t, experts, k, np.random.default_rng(0))[0]))
    return {"bytes": n * (used * expert + t * hidden * 2 * (1 + k)), "flops": n * 2.0 * t * k * 3 * ffn * hidden}


def tolerance(case):
    # four times the error seen against exact(): a linear layer's is its output's own rounding (2.1e-4 in float16,
    # 1.7e-3 in bfloat16); a routed layer's SwiGLU is rounded in steps as well (5.2e-4, 4.3e-3); a whole block's
    # float16 combine adds its own (8.6e-4). float32: the order of the sums
    if case["family"] == "moe":
        return {"rel": 3.5e-3}
    if case["family"] == "glu":
        return {"rel": 2.2e-3 if case["dtype"] == "f16" else 1.7e-2}
    return {"rel": {"f32": 1e-5, "f16": 1.2e-3, "bf16": 7e-3}[case["dtype"]]}


# ---- what the products are in 64 bits, from the formats' definitions

# the codebooks, three bits a value, four values an entry
IQ3_S_GRID = (
    "00000100200500700800900a00c00e01001101501b02002202502702902b03003203903c03f04004104204404804904d"
    "05005305705905d06407107507a08008108508708808b08e09109509809c0a20a50a70a90ab0b80bb0c30c90cd0d00d2"
    "0d90db0de0e40e80ea0f70f90fd10010b10f11111411a12012312913814214415015215615b16116516717617b186189"
    "18b1991aa1b91c01c21c41d01d21d61db1e81ec20020120220420820920b20d20f21021221921c21e22c22e23123a240"
    "24124324624824c25125825b26126826a27827e28028a28d28f29029429a2a02a32ad2b02ba2c12c42c72c82cb2d12d7"
    "2d82dc2e12f22f830330530a30c31931b32232632832c34134834b35135835a3693903943973a43a63c13c33c83ca3d1"
    "3dd3e13f23f840040140340540740840a40c40e41141341741841a42142342542842a43743843b43d44044244844b44f"
    "45245545945c46246948148448749149349849f4a14ab4af4b94bc4c04c24c54c94d24d44d94db4e24e84f6501507510"
    "51351a51d52153a53d54454955255f56056b5785805825875915ad5b15c55c95d65d85e35e860260960b60d60f612619"
    "61b61d62262462762963363964164364564c65165366067067a67e68068a69069a69c6a86c16c86cc6d16d36d76d86e1"
    "6e36e76ed6fb70370970e71271972a73073474174874a75575a76476e77b78e7a17c17c37d07d27dd80080480a810814"
    "81781a82182883884284784984b85285885d86386986d88188388888d89189b8a08af8b28b88c48c98cb8d08d28d98dd"
    "90090291491f92093994594795197298b99c9b09c89cd9d89e39e9a02a08a0ca12a20a24a27a2aa36a3ca41a43a45a4a"
    "a51a5aa7aa80a89a93a98a9eaabac2ac7ac8ad7ae4ae9af5afbb01b04b10b1ab26b4ab56b69b6bba2bc2bc4bd2c09c0b"
    "c0dc19c1bc30c40c50c57c74c8ac9cca2cadcb2cb8cc0ccccd1ce0d15d23d32d40d43d5cd70d85da0dc9dcbe00e04e07"
    "e10e12e1ee20e2ce32e42e49e54e63e65e81e84e88e8ee91e98ea9ec2edaeddeebf01f05f0bf10f28f52f62f82f99fc0")
IQ3_XXS_GRID = (
    "00000200400900b00f01001201902203b03d04104304804a05105505805a06106c07808008208408909009209909b09f"
    "0a90af0bd0c10c70c80ca0d50f810b11f12412f13b13d14114715a16a19d1b41c81cc1ce1e31f120120320820a211213"
    "21821a21c22722824024224925025228128328828a2912982ba2c02c22d02d92e62f63013053283503543663793853d2"
    "3e040040240940b41041241641942244144344544844a45145847347747848048248948f49049249f4a04ad4c14c84cc"
    "4f84fc51d52b54355756157c5c15c35ce5e560160860a61161362863563a6406426506596646666816836886956aa6ba"
    "6c96db71872773a74074675276d78c79e7b37db7f080480f81d81f82b82f87c89089f8a08b08b68c78e5904929934955"
    "9639789c59c89ca9d8a0aa21a38a40a46a56a6da8ca9aabaac2aebb08b13b17b3ab42b59ba8bd4be2c14c24c26c34c51"
    "c71c8fcb4cd8cded24d45d6ad9bdc3dd1e03e05e07e08e1ae2ae56e60e8aea5eaaec0ecdedbef0f11f21f40f42f54f98")


def _grid(digits, levels):
    v = torch.tensor([int(digits[i:i + 3], 16) for i in range(0, len(digits), 3)])
    return torch.tensor(levels, dtype=torch.float64)[torch.stack([(v >> (3 * j)) & 7 for j in range(4)], 1)]


_TABLES = {}


def _table(name, device):
    if name not in _TABLES:
        _TABLES[name] = {"IQ3_S": lambda: _grid(IQ3_S_GRID, [1, 3, 5, 7, 9, 11, 13, 15]),
                         "IQ3_XXS": lambda: _grid(IQ3_XXS_GRID, [4, 12, 20, 28, 36, 44, 52, 62]),
                         "IQ4_NL": lambda: torch.tensor([-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69,
                                                         89, 113], dtype=torch.float64)}[name]().to(device)
    return _TABLES[name]


def _half(b, at):
    return b[:, at:at + 2].contiguous().view(torch.float16).double()


def _bits(v, shifts, mask):
    return (v[..., None] >> torch.tensor(shifts, device=v.device)) & mask


def _weights(blocks, kind, rows, cols):
    """The weights (rows, cols) of a matrix's blocks in float64."""
    per, size = BLOCK[kind]
    b = blocks[:rows * cols // per * size].reshape(-1, size)
    n, dev = b.shape[0], b.device
    if kind == "Q2_0":
        w = _half(b, 0) * (_bits(b[:, 2:].int(), [0, 2, 4, 6], 3).reshape(n, 64) - 1)
    elif kind == "IQ4_NL":
        q = b[:, 2:].long()
        w = _half(b, 0) * _table(kind, dev)[torch.cat([q & 15, q >> 4], 1)]
    elif kind == "Q8_0":
        w = _half(b, 0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif kind == "Q4_K":
        p = b[:, 4:16].int()
        sc = torch.cat([p[:, :4] & 63, (p[:, 8:] & 15) | ((p[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([p[:, 4:8] & 63, (p[:, 8:] >> 4) | ((p[:, 4:8] >> 6) << 4)], 1)
        q = b[:, 16:].int().reshape(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32)
        w = q * (_half(b, 0) * sc)[..., None] - (_half(b, 2) * mn)[..., None]
    elif kind == "Q6_K":
        ql, qh = b[:, :128].int().reshape(n, 2, 2, 32), b[:, 128:192].int().reshape(n, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)
        high = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * _half(b, 208)
        w = ((low | (high << 4)) - 32).reshape(n, 16, 16) * sc[..., None]
    else:
        d = _half(b, 0)
        if kind == "IQ3_S":
            high = _bits(b[:, 66:74].int(), list(range(8)), 1).reshape(n, 64)
            sign = _bits(b[:, 74:106].int(), list(range(8)), 1).reshape(n, 8, 32)
            scale = d * (1 + 2 * _bits(b[:, 106:110].int(), [0, 4], 15).reshape(n, 8))
            index = b[:, 2:66].long() | (high.long() << 8)
        else:
            aux = b[:, 66:98].contiguous().reshape(-1).view(torch.int32).reshape(n, 8).long() & 0xffffffff
            seven = _bits(aux, [0, 7, 14, 21], 127)
            bits = _bits(seven, list(range(7)), 1)
            sign = torch.cat([bits, bits.sum(-1, keepdim=True) & 1], -1).reshape(n, 8, 32)
            scale = d * (0.5 + (aux >> 28).double()) * 0.5
            index = b[:, 2:66].long()
        w = (_table(kind, dev)[index].reshape(n, 8, 32) * (1 - 2 * sign)) * scale[..., None]
    return w.reshape(rows, cols)


def _expert(stack, kind, rows, cols, e):
    size = rows * _row_bytes(kind, cols)
    return _weights(stack[e * size:(e + 1) * size], kind, rows, cols)


def _swiglu(x, gate, up):
    g = x @ gate.T
    return g * torch.sigmoid(g) * (x @ up.T)


def _routed(p, idx, gate, down, ffn, hidden):
    x = p["x"].double()
    y = torch.zeros((*idx.shape, hidden), dtype=torch.float64, device=x.device)
    for e in torch.unique(idx).tolist():
        t, s = torch.nonzero(idx == e, as_tuple=True)
        h = _swiglu(x[t], _expert(p["gate"], gate, ffn, hidden, e), _expert(p["up"], gate, ffn, hidden, e))
        y[t, s] = h @ _expert(p["down"], down, hidden, ffn, e).T
    return y


def exact(case, seed):
    outs = []
    for p in _parts(case, seed):
        x = p["x"].double()
        if case["family"] == "linear":
            rows, cols = case["rows"], case["cols"]
            part = 16384  # rows at a time
            step = _row_bytes(case["kind"], cols)
            outs.append(torch.cat([x @ _weights(p["w"][r * step:(r + part) * step], case["kind"], min(part, rows - r),
                                                cols).T for r in range(0, rows, part)], 1))
            continue
        moe = case["family"] == "moe"
        experts, k, ffn, hidden = SHAPES["a" if moe else case["shape"]]
        if not moe:
            outs.append(_routed(p, p["idx"], case["gate"], case["down"], ffn, hidden))
            continue
        logits, idx = torch.topk(x @ p["router"].double().T, k, dim=1)
        y = (_routed(p, idx, "IQ3_S", "IQ3_S", ffn, hidden) * torch.softmax(logits, 1)[..., None]).sum(1)
        h = _swiglu(x, _weights(p["shared_gate"], "Q4_K", ffn, hidden), _weights(p["shared_up"], "Q4_K", ffn, hidden))
        s = h @ _weights(p["shared_down"], "Q4_K", hidden, ffn).T
        outs.append(y + torch.sigmoid(x @ p["shared_expert_gate"].double().T) * s)
    return outs if case["layers"] else outs[0]
