"""The measured cases: what a program that runs a trellis-packed model has this package do.

A case is one layer or one group of layers called through the package's public entry points
(PackedLinear, PackedGroup, TrellisLinear, PackedLinear.embed_rows, encode_tiles), with the
weights resident on the GPU, as a serving loop holds them. The sizes are those of the
benchmark and the tests: SmolLM2's up projection, the Qwen3-8B block's linears (q 4096x4096,
k/v 1024x4096, o 4096x4096, gate/up 12288x4096, down 4096x12288) and its 4-bit head
(151936x4096), plus a generic size that is a multiple of 16 and of nothing larger.
"""
from __future__ import annotations

import functools
import importlib
import math

import torch

te = importlib.import_module("trellis-everywhere_amd")

DEV = "cuda"
MUL_ADD = {"mcg": (0xCBAC1FED, 0), "3inst": (89226354, 64248484), "1mad": (34038481, 76625530)}
DTYPES = {"f16": torch.float16, "f32": torch.float32, "bf16": torch.bfloat16}
QKV, O, GATE_UP, DOWN = "4096x4096+1024x4096+1024x4096", "4096x4096", "12288x4096+12288x4096", "4096x12288"


def _linear(name, shapes, batch, **more):
    """`shapes`: the members' n x k, joined by + (one: a PackedLinear, several: a PackedGroup)."""
    c = {"name": name, "kind": "linear", "shapes": shapes, "batch": batch, "K": 3, "V": 1,
         "codebook": "mcg", "x": "f16", "y": "f32", "mma_f16": False}
    c.update(more)
    return c


def listed():
    return [
        # the smallest call: one token through one layer of a small model, where the call itself counts
        _linear("small_b1", "1536x576", 1, codebook="3inst", x="f32"),
        # one decoded token: the widest launch of an 8B block (two matrices on one input)
        _linear("gate_up_b1", GATE_UP, 1),
        # one decoded token as it is served: four blocks' seven linears each (qkv, o, gate/up,
        # down: four launches a block) captured in a HIP graph and replayed; the weights of
        # four blocks and three such states do not fit the GPU's last-level cache
        {"name": "blocks_b1", "kind": "blocks", "blocks": 4, "batch": 1, "K": 3, "V": 1, "codebook": "mcg"},
        # the largest matrix of a decoded token: the 4-bit head, f32 logits
        _linear("head_b1", "151936x4096", 1, K=4),
        # a few sequences decoded together, or a draft of four tokens checked
        _linear("down_b4", DOWN, 4, y="f16"),
        # a small serving batch on the narrow group
        _linear("qkv_b16", QKV, 16),
        # a larger serving batch (decode of 64 sequences) on the wide group
        _linear("gate_up_b64", GATE_UP, 64, y="f16"),
        # a ragged layer through the torch.nn adapter: bf16 activations, a bias, odd sizes
        # (Hadamard blocks of 16 and 32), two weights a step
        {"name": "ragged_b37", "kind": "module", "shapes": "1376x2000", "batch": 37, "K": 2, "V": 2,
         "codebook": "3inst", "x": "bf16", "bias": True, "mma_f16": False},
        # a prompt of 512 tokens in the default (exact) mode, the group that takes half of a block
        _linear("prefill_gate_up_512", GATE_UP, 512),
        # a long prompt in the fp16-weight mode a program opts into for prefill, at four bits
        _linear("prefill_down_2048_f16", DOWN, 2048, K=4, y="f16", mma_f16=True),
        # a prompt's embedding rows from the 4-bit table
        {"name": "embed_512", "kind": "embed", "shapes": "151936x4096", "tokens": 512, "K": 4, "V": 1,
         "codebook": "mcg", "y": "f16"},
        # quantizing: the tail-biting encoder over a slice of a layer
        {"name": "encode_1024", "kind": "encode", "tiles": 1024, "K": 3, "codebook": "mcg"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["group"] * 2 + ["module", "embed", "encode"])
    c = {"K": rng.choice([2, 3, 3, 4]), "V": rng.choice([1, 1, 1, 2]),
         "codebook": rng.choice(["mcg", "mcg", "3inst", "1mad"])}
    if kind == "encode":
        del c["V"]
        return {"kind": "encode", "tiles": _log_int(rng, 16, 1024), **c}

    def dim(lo, hi):
        # multiples of 16 over the range, half of them of 128 (a full Hadamard block)
        step = rng.choice([16, 128])
        return max(1, _log_int(rng, lo, hi) // step) * step

    if kind == "embed":
        return {"kind": "embed", "shapes": "%dx%d" % (dim(4096, 151936), dim(512, 4096)),
                "tokens": _log_int(rng, 1, 512), "y": rng.choice(["f16", "f32"]), **c}
    k = dim(512, 12288)
    count = rng.choice([2, 3]) if kind == "group" else 1
    ns = [dim(512, 12288) for _ in range(count)]
    # rows of activations: one to a long prompt, at most the largest listed case's products
    most = int(1e11 // (k * sum(ns)))
    c.update(shapes="+".join("%dx%d" % (n, k) for n in ns), batch=_log_int(rng, 1, max(1, min(2048, most))),
             mma_f16=rng.random() < 0.3)
    if kind == "module":
        return {"kind": "module", "x": rng.choice(["f16", "bf16"]), "bias": rng.random() < 0.5, **c}
    return {"kind": "linear", "x": rng.choice(["f16", "f16", "f32"]), "y": rng.choice(["f16", "f32"]), **c}


def _members(case):
    if case["kind"] == "blocks":
        return [m for _ in range(case["blocks"]) for g in (QKV, O, GATE_UP, DOWN) for m in _parse(g)]
    return _parse(case["shapes"])


def _parse(shapes):
    return [tuple(int(v) for v in s.split("x")) for s in shapes.split("+")]


def _tensors(case, seed):
    """Everything a case is made of, from its seed alone: the members' packed words, signs and
    scales (uniform random words are what an encoder's output looks like) and the inputs."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)

    def uniform(n):   # per-channel scales, fp16 on disk, mean about 1
        return (torch.rand(n, generator=g, device=DEV) + 0.5).half().float()

    def signs(n):
        return torch.randint(0, 2, (n,), generator=g, device=DEV).float() * 2 - 1

    out = {"members": []}
    if case["kind"] == "encode":
        # z-space targets: unit normal after the incoherence transform
        out["w"] = torch.randn((case["tiles"], 256), generator=g, device=DEV)
        return out
    for n, k in _members(case):
        bits = torch.randint(-2 ** 31, 2 ** 31 - 1, (n // 16 * (k // 16), 8 * case["K"]), generator=g,
                             device=DEV, dtype=torch.int32)
        out["members"].append({"n": n, "k": k, "bits": bits, "su": signs(k), "sv": signs(n),
                               "isc": uniform(k) * 0.016, "osc": uniform(n)})
    if case["kind"] == "embed":
        out["tokens"] = torch.randint(0, out["members"][0]["n"], (case["tokens"],), generator=g,
                                      device=DEV).int()
    elif case["kind"] == "blocks":
        # each block's inputs of the four launches, ready as the rest of the model leaves them
        out["x"] = [[torch.randn((case["batch"], k), generator=g, device=DEV).half()
                     for k in (4096, 4096, 4096, 12288)] for _ in range(case["blocks"])]
    else:
        out["x"] = torch.randn((case["batch"], out["members"][0]["k"]), generator=g,
                               device=DEV).to(DTYPES[case["x"]])
        if case.get("bias"):
            out["bias"] = torch.randn(out["members"][0]["n"], generator=g, device=DEV)
    return out


def _packed(case, m):
    return te.PackedLinear.from_device(m["n"], m["k"], case["K"], m["bits"], m["su"], m["sv"], m["isc"],
                                       m["osc"], codebook=case["codebook"], V=case["V"])


def prepare(case, seed):
    t = _tensors(case, seed)
    kind = case["kind"]
    if kind == "encode":
        return {"call": lambda: te.encode_tiles(t["w"], case["K"], case["codebook"])}
    lins = [_packed(case, m) for m in t["members"]]
    if kind == "embed":
        return {"call": lambda: lins[0].embed_rows(t["tokens"], out_dtype=DTYPES[case["y"]])}
    if kind == "module":
        layer = te.TrellisLinear(lins[0], bias=t.get("bias"), mma_f16=case["mma_f16"])
        return {"call": lambda: layer(t["x"])}
    if kind == "blocks":
        return _captured_blocks(case, lins, t["x"])
    y, mma = DTYPES[case["y"]], case["mma_f16"]
    # the workspace is sized once when a model is loaded
    if len(lins) == 1:
        lins[0].reserve(case["batch"])
        return {"call": lambda: lins[0].forward(t["x"], out_dtype=y, mma_f16=mma)}
    group = te.PackedGroup(lins)
    group.reserve(case["batch"])
    xs = [t["x"]] * len(lins)
    return {"call": lambda: group.forward(xs, out_dtype=y, mma_f16=mma)}


def _captured_blocks(case, lins, xs):
    launches, outs = [], []
    for b in range(case["blocks"]):
        q, k, v, o, gate, up, down = lins[7 * b:7 * b + 7]
        for members, x in zip(((q, k, v), (o,), (gate, up), (down,)), xs[b]):
            ys = [torch.empty((case["batch"], m.n_out), device=DEV) for m in members]
            group = te.PackedGroup(members)
            group.reserve(case["batch"])
            launches.append((group, [x] * len(members), ys))
            outs += ys

    def step():
        for group, x, ys in launches:
            group.forward(x, outs=ys)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()

    def replay():
        graph.replay()
        return outs

    return {"call": replay, "keep": launches}


def run(state):
    return state["call"]()


def work(case):
    kind = case["kind"]
    if kind == "encode":
        # two passes over 256 steps, 2^16 states a step, three operations a state
        return {"bytes": case["tiles"] * (256 * 8 + 32 * case["K"]), "flops": case["tiles"] * 2 * 256 * 65536 * 3}
    members = _members(case)
    if kind == "embed":
        n, k = members[0]
        t = case["tokens"]
        # each token's row needs the weights of its row's Hadamard block (counted once where
        # tokens share one), one multiply-add each
        rows = _fit(n)
        blocks = n // rows
        distinct = blocks * (1 - (1 - 1 / blocks) ** t)
        return {"bytes": distinct * rows * k * case["K"] / 8 + t * (k * _size(case["y"]) + 4) + 8 * k,
                "flops": 2 * t * rows * k}
    b = case["batch"]
    nbytes = sum(n * k * case["K"] / 8 + 8 * (n + k) for n, k in members)
    flops = sum(2 * b * n * k for n, k in members)
    x, y = case.get("x", "f16"), case.get("y", case.get("x", "f32") if kind == "module" else "f32")
    inputs = sum(b * k for k in (4096, 4096, 4096, 12288)) * case["blocks"] if kind == "blocks" else b * members[0][1]
    nbytes += inputs * _size(x) + sum(b * n for n, _ in members) * _size(y)
    return {"bytes": nbytes, "flops": flops}


def _size(dtype):
    return 4 if dtype == "f32" else 2


def tolerance(case):
    if case["kind"] == "encode":
        return "exact"    # whole words, and codebook values copied
    if case["kind"] == "embed":
        # fp32 sums of exact weights; f16 rows are rounded once
        return {"rel": 1e-3, "max": 4e-3} if case["y"] == "f16" else {"rel": 2e-6, "max": 2e-5}
    if case.get("x") == "bf16":
        return {"rel": 8e-3, "max": 4e-2}     # the output is rounded to bf16
    # the folded activations are rounded to fp16 (and the weights in the fp16-weight mode),
    # sums and folds in fp32: about 2e-4 against exact sums, 3e-4 in the fp16-weight mode
    return {"rel": 1e-3, "max": 6e-3}


# ---------------------------------------------------------------- 64-bit values
def _fit(d):
    return math.gcd(d, 128)


@functools.lru_cache(maxsize=None)
def _hadamard(d):
    h = torch.ones((1, 1), dtype=torch.float64, device=DEV)
    while h.shape[0] < d:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(d)


def _block_had(v, d):
    """Normalized block-diagonal Hadamard over the last axis, blocks of d."""
    return (v.reshape(-1, d) @ _hadamard(d)).reshape(v.shape)


def _decode(bits, K, V, codebook):
    """Packed words [tiles, 8K] -> float64 [tiles, 256] in tile order (row, column)."""
    mul, add = MUL_ADD[codebook]
    words = bits.long() & 0xFFFFFFFF
    step = K * V
    at = (256 // V - 1 - torch.arange(256 // V, device=DEV)) * step
    lo, hi = words[:, at >> 5], words[:, ((at >> 5) + 1) % (8 * K)]
    state = ((lo | (hi << 32)) >> (at & 31)) & 0xFFFF
    p = [(state * mul + add) & 0xFFFFFFFF]
    if V == 2:
        p.append((p[0] * mul + add) & 0xFFFFFFFF)
    p = torch.stack(p, -1).reshape(bits.shape[0], 256)
    if codebook == "1mad":
        y = (p & 255) + (p >> 8 & 255) + (p >> 16 & 255) + (p >> 24)
        return (y.double() - 510) / 147.800537109375
    p = (p & 0x8FFF8FFF) ^ 0x3B603B60

    def half(v):   # the low 16 bits as an fp16 number
        return ((v & 0xFFFF) - ((v & 0x8000) << 1)).to(torch.int16).view(torch.float16).double()

    return half(p >> 16) + half(p)


def _rows(case, m, r0, r1):
    """z-space rows r0 .. r1 - 1 (multiples of 16) of a member, float64 [r1 - r0, k]."""
    tin = m["k"] // 16
    z = _decode(m["bits"][r0 // 16 * tin:r1 // 16 * tin], case["K"], case["V"], case["codebook"])
    return z.view((r1 - r0) // 16, tin, 16, 16).transpose(1, 2).reshape(r1 - r0, m["k"])


def _exact_linear(case, m, x):
    xf = _block_had(x.double() * m["isc"].double() * m["su"].double(), _fit(m["k"]))
    t = torch.empty((x.shape[0], m["n"]), dtype=torch.float64, device=DEV)
    for r in range(0, m["n"], 2048):
        e = min(m["n"], r + 2048)
        t[:, r:e] = xf @ _rows(case, m, r, e).t().contiguous()
    return _block_had(t, _fit(m["n"])) * m["sv"].double() * m["osc"].double()


def _exact_embed(case, m, tokens):
    d = _fit(m["n"])
    out = []
    for r in tokens.tolist():
        z = _rows(case, m, r // d * d, r // d * d + d)
        w = (_hadamard(d)[r % d][None] @ z)[0]
        out.append(_block_had(w, _fit(m["k"])) * m["su"].double() * m["isc"].double()
                   * m["sv"][r].double() * m["osc"][r].double())
    return torch.stack(out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "encode":
        return None       # whole words; the path's ties are those of its fp32 sums
    t = _tensors(case, seed)
    if kind == "embed":
        return _exact_embed(case, t["members"][0], t["tokens"])
    if kind == "blocks":
        ys = []
        for i, m in enumerate(t["members"]):
            launch = (0, 0, 0, 1, 2, 2, 3)[i % 7]
            ys.append(_exact_linear(case, m, t["x"][i // 7][launch]))
        return ys
    ys = [_exact_linear(case, m, t["x"]) for m in t["members"]]
    if kind == "module":
        return ys[0] + t["bias"].double() if "bias" in t else ys[0]
    return ys[0] if len(ys) == 1 else ys
