"""The workloads that this library's speed is judged by.

A decode engine calls the library in a handful of ways: projections of one token or of a
verifier's block of up to sixteen, whole layers of them with the norms and the attention in
between, the vocabulary projection with its argmax, and prompts of any length through the prefill
GEMM or the exact linear.  `listed()` names twelve such calls at the sizes that the tests and the
benchmark use (model width 6,656, 32 query heads over 2 key/value heads of 128, feed-forward width
16,384, vocabulary 202,048); `draw()` gives others from the same ranges, odd sizes among them.

Weights are quantized from N(0, 0.02) by the library's own quantizer: a pool of 2,048 blocks per
format, from which every tensor takes its blocks at random, so that tensors of a gigabyte are made
in milliseconds and hold the codes and scales of real ones.  Activations are N(0, 1) rounded to
bf16; cache rows are bf16 N(0, 1); norm weights lie around one.
"""
from __future__ import annotations

import math

import torch

from neuralfn_amd import decode_layer as dl
from neuralfn_amd import engine_ops, kquant, tile_ops

ENCODINGS = {"f32": kquant.F32, "bf16": kquant.BF16, "q8_0": kquant.Q8_0, "q4_k": kquant.Q4_K,
             "q5_k": kquant.Q5_K, "q6_k": kquant.Q6_K}
PACKED = ("q4_k", "q5_k", "q6_k", "q8_0")
HEAD_DIM = 128
DEVICE = "cuda:0"

MODEL = {"width": 6656, "heads": 32, "kv_heads": 2}
FFN = 16384
VOCABULARY = 202048


def listed():
    return [
        # one layer's attention projections (Q, K and V in one call, then O) of one token: the
        # smallest calls a decode step makes, bound by launches
        dict(MODEL, name="projections_1_layer", kind="projections", encoding="q4_k", rows=1, layers=1, graph=False),
        # the same projections of a whole 48-layer step, captured once and replayed per token
        dict(MODEL, name="projections_48_layers", kind="projections", encoding="q4_k", rows=1, layers=48, graph=True),
        # one decode step of eight local layers (2,048-key window), captured and replayed
        dict(MODEL, name="decode_8_layers", kind="decode", encoding="q4_k", down="q6_k", ffn=FFN, layers=8,
             keys=2048, local=True, graph=True),
        # one token through two global layers deep into a long context, called operator by operator
        dict(MODEL, name="decode_long_context", kind="decode", encoding="q5_k", down="q6_k", ffn=FFN, layers=2,
             keys=32768, local=False, graph=False),
        # a speculative block of seven tokens through four layers, every row as the one-token call
        # computes it
        dict(MODEL, name="verify_7_rows", kind="verify", encoding="q4_k", down="q6_k", ffn=FFN, layers=4, rows=7,
             keys=2048, local=True, family="mmvq", graph=False),
        # the feed-forward projections of a full block of sixteen (a prompt's 16-token chunk)
        dict(MODEL, name="ffn_16_rows", kind="ffn", encoding="q4_k", down="q6_k", ffn=FFN, rows=16, family="mmq"),
        # the next token's index: vocabulary projection and argmax, for one token and for a block
        dict(name="lm_head_1_row", kind="lm_head", encoding="q6_k", width=6656, vocabulary=VOCABULARY, rows=1),
        dict(name="lm_head_16_rows", kind="lm_head", encoding="q6_k", width=6656, vocabulary=VOCABULARY, rows=16),
        # a short prompt of no round length through a layer's attention inputs (Q, K, V, gate)
        dict(MODEL, name="prefill_333_attention", kind="prefill", part="attention", encoding="q5_k", ffn=FFN, rows=333),
        # a prompt of 2,048 tokens through the down projection
        dict(MODEL, name="prefill_2048_down", kind="prefill", part="down", encoding="q6_k", ffn=FFN, rows=2048),
        # a long prompt through gate and up, the largest call
        dict(MODEL, name="prefill_4096_gate_up", kind="prefill", part="gate_up", encoding="q4_k", ffn=FFN, rows=4096),
        # the exact linear (any format, float arithmetic) with a bias, for a caller without the GEMM's workspace
        dict(name="exact_linear_200_rows", kind="linear", encoding="q8_0", width=4096, out=6656, rows=200, bias=True),
    ]


def draw(rng):
    def spread(low, high):
        return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))))

    def blocks(low, high):  # packed rows are whole blocks of 256 values
        return 256 * rng.randint(low // 256, high // 256)

    kind = rng.choice(("projections", "decode", "verify", "ffn", "lm_head", "prefill", "linear"))
    model = {"width": blocks(2048, 8192), "heads": rng.choice((16, 32, 48)), "kv_heads": rng.choice((2, 4, 8))}
    ffn, encoding, down = blocks(4096, 19968), rng.choice(PACKED), rng.choice(PACKED)
    family, graph = rng.choice(("mmq", "mmvq")), rng.random() < 0.5
    if kind == "projections":
        return dict(model, kind=kind, encoding=encoding, rows=spread(1, 16), layers=spread(1, 48), graph=graph)
    if kind == "decode":
        return dict(model, kind=kind, encoding=encoding, down=down, ffn=ffn, layers=rng.randint(1, 8),
                    keys=spread(100, 32768), local=rng.random() < 0.5, graph=graph)
    if kind == "verify":
        return dict(model, kind=kind, encoding=encoding, down=down, ffn=ffn, layers=rng.randint(1, 4),
                    rows=rng.randint(2, 16), keys=spread(100, 8192), local=rng.random() < 0.5, family=family, graph=graph)
    if kind == "ffn":
        return dict(model, kind=kind, encoding=encoding, down=down, ffn=ffn, rows=rng.randint(1, 16), family=family)
    if kind == "lm_head":
        return dict(kind=kind, encoding=rng.choice(PACKED[:3]), width=model["width"],
                    vocabulary=spread(4000, VOCABULARY), rows=spread(1, 16))
    if kind == "prefill":
        case = dict(model, kind=kind, part=rng.choice(("attention", "output", "gate_up", "down")), encoding=encoding,
                    ffn=ffn, rows=spread(17, 4096))
        weights = sum(out * width for out, width in _prefill_shapes(case))
        return dict(case, rows=min(case["rows"], 4096 * 2 * FFN * MODEL["width"] // weights))  # no larger than the largest
    return dict(kind=kind, encoding=rng.choice(PACKED + ("bf16", "f32")), width=model["width"], out=spread(64, 8192),
                rows=spread(1, 512), bias=rng.random() < 0.5)


# -- inputs ------------------------------------------------------------------------------------


class _Maker:
    """Weights and activations from one seed."""

    def __init__(self, seed: int):
        self.seed = seed
        self.generator = torch.Generator(device=DEVICE).manual_seed(seed)
        self.pools = {}

    def normal(self, *shape):
        return torch.randn(shape, generator=self.generator, device=DEVICE)

    def activations(self, rows: int, width: int):
        return self.normal(rows, width).to(torch.bfloat16).float()

    def weight(self, encoding: str, out_dim: int, in_dim: int):
        code = ENCODINGS[encoding]
        if encoding in ("f32", "bf16"):
            values = self.normal(out_dim, in_dim) * 0.02
            data = values if encoding == "f32" else values.to(torch.bfloat16)
            return tile_ops.PackedWeight(code, out_dim, in_dim, data.reshape(-1).view(torch.uint8))
        if encoding not in self.pools:
            nbytes = 256 // kquant.BLOCKS[code][0] * kquant.BLOCKS[code][1]
            packed = kquant.quantize(code, kquant.synthetic_weights(self.seed, 512, 1024))
            self.pools[encoding] = torch.from_numpy(packed.reshape(-1, nbytes)).to(DEVICE)
        pool = self.pools[encoding]
        chosen = torch.randint(0, pool.shape[0], (out_dim * in_dim // 256,), generator=self.generator, device=DEVICE)
        return tile_ops.PackedWeight(code, out_dim, in_dim, pool.index_select(0, chosen).reshape(-1))

    def norm(self, width: int):
        return tile_ops.PackedWeight(kquant.F32, 1, width, (1.0 + 0.1 * self.normal(width)).view(torch.uint8))

    def cache(self, geometry):
        cache = dl.LayerCache(geometry, DEVICE)
        for ring in (cache.keys, cache.values):
            ring.copy_(self.normal(*ring.shape).to(torch.bfloat16).view(torch.int16))
        return cache


def _attention_shapes(case):
    """(output width, input width) of Q, K, V and of the attention gate and O."""
    width, q, kv = case["width"], case["heads"] * HEAD_DIM, case["kv_heads"] * HEAD_DIM
    return {"q": (q, width), "k": (kv, width), "v": (kv, width), "attention_gate": (q, width), "output": (width, q)}


def _layers(case, make):
    geometry = dl.LayerGeometry(case["width"], case["heads"], case["kv_heads"], HEAD_DIM, case["ffn"], case["keys"])
    ffn, width = case["ffn"], case["width"]
    weights, caches = [], []
    for _ in range(case["layers"]):
        packed = {name: make.weight(case["encoding"], *shape) for name, shape in _attention_shapes(case).items()}
        weights.append(dl.LayerWeights(
            **packed, mlp_gate=make.weight(case["encoding"], ffn, width), mlp_up=make.weight(case["encoding"], ffn, width),
            mlp_down=make.weight(case["down"], width, ffn), input_norm=make.norm(width), q_norm=make.norm(HEAD_DIM),
            k_norm=make.norm(HEAD_DIM), post_attention_norm=make.norm(width), pre_feedforward_norm=make.norm(width),
            post_feedforward_norm=make.norm(width)))
        caches.append(make.cache(geometry))
    rows = case.get("rows", 1)
    return {"geometry": geometry, "weights": weights, "caches": caches, "x": make.activations(rows, width),
            "zeros": torch.zeros((rows, width), device=DEVICE), "local": case["local"],
            # a local layer is far into its ring, a global one sees every key of the context so far
            "position": case["keys"] + 5000 if case["local"] else case["keys"] - rows,
            "workspace": tile_ops.small_batch_workspace(rows, max(width, ffn, case["heads"] * HEAD_DIM), DEVICE),
            "attention_workspace": engine_ops.gqa_decode_workspace(case["heads"], HEAD_DIM, DEVICE),
            "cached": [ring.view(torch.bfloat16) for cache in caches for ring in (cache.keys, cache.values)]}


def prepare(case, seed):
    make, kind, rows = _Maker(seed), case["kind"], case.get("rows", 1)
    state = {"kind": kind, "rows": rows}
    if kind == "projections":
        shapes = _attention_shapes(case)
        # one buffer per projection holds every layer's outputs
        state["projected"] = {name: torch.zeros((case["layers"], rows, shapes[name][0]), device=DEVICE)
                              for name in ("q", "k", "v", "output")}
        out = {name: list(buffer) for name, buffer in state["projected"].items()}
        state["layers"] = [([make.weight(case["encoding"], *shapes[name]) for name in ("q", "k", "v")],
                            [make.weight(case["encoding"], *shapes["output"])],
                            [out[name][layer] for name in ("q", "k", "v")], [out["output"][layer]])
                           for layer in range(case["layers"])]
        state["x"] = make.activations(rows, case["width"])
        state["attended"] = make.activations(rows, case["heads"] * HEAD_DIM)
        state["workspace"] = tile_ops.small_batch_workspace(rows, max(case["width"], case["heads"] * HEAD_DIM), DEVICE)
    elif kind in ("decode", "verify"):
        state.update(_layers(case, make), family=case.get("family"))
    elif kind == "ffn":
        state["pair"] = [make.weight(case["encoding"], case["ffn"], case["width"]) for _ in range(2)]
        state["down"] = [make.weight(case["down"], case["width"], case["ffn"])]
        state["x"] = make.activations(rows, case["width"])
        state["workspace"] = tile_ops.small_batch_workspace(rows, max(case["width"], case["ffn"]), DEVICE)
        state["family"] = case["family"]
    elif kind == "lm_head":
        state["weight"] = make.weight(case["encoding"], case["vocabulary"], case["width"])
        state["x"] = make.activations(rows, case["width"])
    elif kind == "prefill":
        state["weights"] = [make.weight(case["encoding"], *shape) for shape in _prefill_shapes(case)]
        state["x"] = make.activations(rows, state["weights"][0].input_dim)
    else:
        state["weight"] = make.weight(case["encoding"], case["out"], case["width"])
        state["x"] = make.activations(rows, case["width"])
        state["bias"] = make.normal(case["out"]) if case["bias"] else None
    if case.get("graph"):  # an engine captures its step once and replays it for every token
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _step(state)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outputs = _step(state)
        state["graph"], state["outputs"] = graph, outputs
    return state


def _prefill_shapes(case):
    shapes, ffn, width = _attention_shapes(case), case["ffn"], case["width"]
    return {"attention": [shapes[name] for name in ("q", "k", "v", "attention_gate")], "output": [shapes["output"]],
            "gate_up": [(ffn, width), (ffn, width)], "down": [(width, ffn)]}[case["part"]]


# -- one pass ----------------------------------------------------------------------------------


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    return _step(state)


def _step(s):
    kind = s["kind"]
    if kind == "projections":
        for inputs, output, qkv, o in s["layers"]:
            tile_ops.multi_linear(inputs, s["x"], s["workspace"], outputs=qkv)
            tile_ops.multi_linear(output, s["attended"], s["workspace"], outputs=o)
        return s["projected"]
    if kind == "decode":
        pending, residual, norm = s["x"], s["zeros"], None
        for weights, cache in zip(s["weights"], s["caches"]):
            pending, residual = dl.decode_layer(
                s["geometry"], weights, cache, pending, residual, norm, s["position"], s["workspace"], s["local"],
                s["attention_workspace"], fused_gate_up=True, fused_input_norm=True)
            norm = weights.post_feedforward_norm
        return [pending, residual] + s["cached"]
    if kind == "verify":
        pending, residual, norm, out = s["x"], s["zeros"], None, []
        for weights, cache in zip(s["weights"], s["caches"]):
            pending, residual, keys, values = dl.verify_layer(
                s["geometry"], weights, cache, pending, residual, norm, s["position"], s["workspace"], s["local"],
                s["attention_workspace"], family=s["family"])
            norm = weights.post_feedforward_norm
            out += [keys, values]
        return [pending, residual] + out
    if kind == "ffn":
        gate, up = tile_ops.multi_linear(s["pair"], s["x"], s["workspace"], family=s["family"])
        (down,) = tile_ops.multi_linear(s["down"], gate, s["workspace"], second=up, family=s["family"], prologue="swiglu")
        return gate, up, down
    if kind == "lm_head":
        return tile_ops.lm_head_argmax(s["weight"], s["x"])
    if kind == "prefill":
        if len(s["weights"]) == 1:
            return tile_ops.gemm(s["weights"][0], s["x"])
        return tile_ops.gemm_multi(s["weights"], s["x"])
    return tile_ops.linear(s["weight"], s["x"], s["bias"])


# -- what a pass cannot do without, and how far two correct ones may differ ----------------------


def work(case):
    kind, rows = case["kind"], case.get("rows", 1)
    layers = case.get("layers", 1)
    extra = 0.0
    if kind == "projections":
        shapes = _attention_shapes(case)
        matrices = [(case["encoding"], shapes[name]) for name in ("q", "k", "v", "output")]
        vectors = rows * (case["width"] + sum(shape[0] for _, shape in matrices) + shapes["output"][1])
    elif kind in ("decode", "verify"):
        ffn, width, kv = case["ffn"], case["width"], case["kv_heads"] * HEAD_DIM
        matrices = [(case["encoding"], shape) for shape in _attention_shapes(case).values()]
        matrices += [(case["encoding"], (ffn, width))] * 2 + [(case["down"], (width, ffn))]
        vectors = rows * (3 * width + 2 * kv)
        extra = 2 * 2.0 * kv * case["keys"] + 4.0 * (4 * width + 2 * HEAD_DIM)
    elif kind == "ffn":
        matrices = [(case["encoding"], (case["ffn"], case["width"]))] * 2 + [(case["down"], (case["width"], case["ffn"]))]
        vectors = rows * (2 * case["width"] + 2 * case["ffn"])
    elif kind == "lm_head":
        matrices, vectors = [(case["encoding"], (case["vocabulary"], case["width"]))], rows * (case["width"] + 3)
    elif kind == "prefill":
        shapes = _prefill_shapes(case)
        matrices = [(case["encoding"], shape) for shape in shapes]
        vectors = rows * (shapes[0][1] + sum(shape[0] for shape in shapes))
    else:
        matrices = [(case["encoding"], (case["out"], case["width"]))]
        vectors = rows * (case["width"] + case["out"]) + (case["out"] if case["bias"] else 0)
    nbytes = sum(kquant.packed_nbytes(ENCODINGS[name], *shape) for name, shape in matrices) + 4.0 * vectors + extra
    flops = sum(2.0 * rows * shape[0] * shape[1] for _, shape in matrices)
    if kind in ("decode", "verify"):
        flops += 4.0 * rows * case["heads"] * HEAD_DIM * case["keys"]
    return {"bytes": layers * nbytes, "flops": layers * flops}


def tolerance(case):
    kind, rows = case["kind"], case.get("rows", 1)
    if kind == "linear":  # float products, float sums
        return {"rel": 1e-5, "max": 1e-4}
    if kind in ("decode", "verify"):  # chains of layers; new cache rows are rounded to bf16
        return {"rel": 3e-3, "max": 3e-2}
    if kind == "prefill" or rows > 1 and case.get("family", "mmq") == "mmq":  # fp16 operands
        tolerated = {"rel": 1e-3, "max": 1e-2}
    else:  # 16-bit codes of the activations, exact weights
        tolerated = {"rel": 1e-4, "max": 1e-3}
    return dict(tolerated, differ=0.01) if kind == "lm_head" else tolerated
