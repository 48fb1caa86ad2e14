"""The work that is timed: what a program built on this package has it do, through its public entry points.

A decoder layer's quantized products with the launches that consume them (`layer`), one product alone (`product`), the
vocabulary head with its argmax (`head`) and the trainer's dequantization of a stored matrix (`dequant`). `listed` names
twelve of them, `draw` gives others of the same ranges.

A layer is the sequence the engine runs on one normed input x: the attention in-projection as whole rows; the
out-projection of the attention's output, its partials added to the residual stream h and normed (add_rmsnorm); [gate;
up] with the SwiGLU epilogue; the down projection and the second residual step. Steps of up to 48 tokens (decode,
verification of drafted tokens, batches of sequences) are captured once into a graph and replayed, as a decode loop
does; longer ones (prompts) are launched call by call. With an adapter (`rank`), the stacked A products run first and
their delta is added in the epilogue of [gate; up] and down."""

import math

import numpy as np
import torch

from qwenny_amd import Epi, Gemm, Graph, Mat, Quant, add_rmsnorm, dequant, sum_parts

EPS = 1e-6
GRAPH_TOKENS = 48  # steps of up to this many tokens are replayed from a graph
WHOLE_TOKENS = 8   # in-projections of up to this many tokens are asked for as whole rows, longer ones are summed
INT_MAX = 2**31 - 1

# Widths of the two model sizes the package is measured on: hidden, in-projection rows, out-projection columns, MLP.
SIZE_4B = {"hidden": 2560, "qkv": 4096, "attn": 4096, "inter": 9728}
SIZE_27B = {"hidden": 5120, "qkv": 6144, "attn": 6144, "inter": 17408}


def layer(name, weights, size, tokens, rank=0):
    return {"name": name, "what": "layer", "weights": weights, **size, "tokens": tokens, "rank": rank}


def listed():
    return [
        # the smallest call: one token through one int4 matrix
        {"name": "product_4b_1", "what": "product", "weights": "i4", "rows": 9728, "cols": 2560, "tokens": 1},
        # a decode step of a small model, int4 with zero points, four sequences at once
        layer("layer_4b_zp_4", "i4z", SIZE_4B, 4),
        # the plain decode step: one sequence, a 27B layer of symmetric int4
        layer("layer_27b_1", "i4", SIZE_27B, 1),
        # verification of four drafted tokens after the accepted one
        layer("layer_27b_5", "i4", SIZE_27B, 5),
        # a batch: four sequences of five tokens
        layer("layer_27b_20", "i4", SIZE_27B, 20),
        # decode with the int8 storage (a scale per row and 128 columns, the load-time default for 16-bit checkpoints)
        layer("layer_27b_int8_1", "i8g", SIZE_27B, 1),
        # 16-bit matrices of a checkpoint, twelve sequences
        layer("layer_4b_bf16_12", "bf16", SIZE_4B, 12),
        # logits and greedy token of a verification step over the 27B vocabulary
        {"name": "head_27b_5", "what": "head", "weights": "i4", "rows": 248320, "cols": 5120, "tokens": 5},
        # a short prompt of a small model
        layer("layer_4b_100", "i4", SIZE_4B, 100),
        # a prompt of ragged length with a rank-16 adapter on the MLP, int4 with zero points
        layer("layer_27b_zp_adapter_333", "i4z", SIZE_27B, 333, rank=16),
        # the largest prefill chunk
        layer("layer_27b_2048", "i4", SIZE_27B, 2048),
        # the trainer's dense rows of one stored matrix
        {"name": "dequant_27b", "what": "dequant", "weights": "i4", "rows": 17408, "cols": 5120, "f32": False},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _multiple(rng, lo, hi, unit):
    return max(lo, min(hi, int(round(_log(rng, lo, hi) / unit)) * unit))


def draw(rng):
    what = rng.choices(("layer", "product", "head", "dequant"), (10, 3, 2, 2))[0]
    if what == "dequant":
        return {"what": what, "weights": rng.choice(("i4", "i4z", "i8g")), "rows": int(_log(rng, 200, 17408)),
                "cols": _multiple(rng, 1024, 5120, 128), "f32": rng.random() < 0.3}
    if what == "product":
        return {"what": what, "weights": rng.choice(("i4", "i4z", "i8g", "i8", "bf16")),
                "rows": _multiple(rng, 512, 17408, 16), "cols": _multiple(rng, 1024, 17408, 128),
                "tokens": int(_log(rng, 1, 513))}
    if what == "head":
        return {"what": what, "weights": rng.choice(("i4", "i4z", "i8g")), "rows": _multiple(rng, 32000, 151936, 16),
                "cols": _multiple(rng, 1024, 5120, 128), "tokens": int(_log(rng, 1, 65))}
    size = {"hidden": _multiple(rng, 1024, 5120, 128), "qkv": _multiple(rng, 1024, 10240, 16),
            "attn": _multiple(rng, 1024, 6144, 128), "inter": _multiple(rng, 2048, 17408, 128)}
    return {"what": what, "weights": rng.choice(("i4", "i4", "i4z", "i4z", "i8g", "i8", "bf16")), **size,
            "tokens": int(_log(rng, 1, 2049)), "rank": rng.choice((0, 0, 0, 8, 16, 64))}


# ---- inputs ---------------------------------------------------------------------------------------------------------


def _gen(seed, name):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1_000_003 + sum((i + 1) * ord(c) for i, c in enumerate(name))) & 0x7FFFFFFFFFFF)
    return g


def _stored(seed, name, weights, rows, cols):
    """One matrix as a checkpoint stores it, on the GPU: (bits, group, words int32 [rows][cols * bits / 32], scales f32
    [rows][groups], zero points int32 [rows][groups]); dense: bf16 [rows][cols]. Scales are bf16 values."""
    g = _gen(seed, name)
    if weights == "bf16":
        return (torch.randn((rows, cols), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    bits = 4 if weights in ("i4", "i4z") else 8
    group = cols if weights == "i8" else 128
    if bits == 4:
        words = torch.randint(-2**31, 2**31, (rows, cols // 8), generator=g, device="cuda", dtype=torch.int64)
        words = words.to(torch.int32)
        lo, hi = 0.002, 0.02
    else:
        words = torch.randint(1, 256, (rows, cols), generator=g, device="cuda", dtype=torch.int16).to(torch.uint8)
        words = words.view(torch.int32)
        lo, hi = 0.0001, 0.001
    scales = torch.rand((rows, cols // group), generator=g, device="cuda") * (hi - lo) + lo
    scales = scales.to(torch.bfloat16).float()
    if weights == "i4z":
        zeros = torch.randint(4, 13, scales.shape, generator=g, device="cuda", dtype=torch.int32)
    else:
        zeros = torch.full(scales.shape, 1 << (bits - 1), dtype=torch.int32, device="cuda")
    return bits, group, words, scales, zeros


def _dense64(stored):
    """The matrix in 64 bits."""
    if isinstance(stored, torch.Tensor):
        return stored.double()
    bits, group, words, scales, zeros = stored
    rows, cols = words.shape[0], words.shape[1] * 32 // bits
    if bits == 8:
        q = words.view(torch.uint8)
    else:
        b = words.view(torch.uint8)
        q = torch.stack((b & 15, b >> 4), -1)
    q = q.reshape(rows, cols // group, group).double()
    return ((q - zeros[..., None]) * scales.double()[..., None]).reshape(rows, cols)


def _host(stored):
    """What a checkpoint reader hands to Mat.stack: a Quant, or (bf16 bits, cols)."""
    if isinstance(stored, torch.Tensor):
        return stored.view(torch.int16).cpu().numpy().view(np.uint16), stored.shape[1]
    bits, group, words, scales, zeros = stored
    return Quant(bits, group, words.shape[0], words.shape[1] * 32 // bits, words.cpu().numpy().view(np.uint32),
                 scales.cpu().numpy(), (-zeros * scales).cpu().numpy())


_GEMM = []


def _gemm():
    """The program's one context."""
    if not _GEMM:
        _GEMM.append(Gemm.load(0))
    return _GEMM[0]


def _mat(stored, silu=False):
    return Mat.stack(_gemm(), [_host(s) for s in stored], silu=silu, int8=False)


def _matrices(case, seed):
    """The layer's matrices as stored, by name."""
    h, w = case["hidden"], case["weights"]
    return {"qkv": _stored(seed, "qkv", w, case["qkv"], h), "out": _stored(seed, "out", w, h, case["attn"]),
            "gate": _stored(seed, "gate", w, case["inter"], h), "up": _stored(seed, "up", w, case["inter"], h),
            "down": _stored(seed, "down", w, h, case["inter"])}


def _activations(seed, name, tokens, cols):
    """bf16 N(0, 1); in prompts 1 % of the columns are outliers (x 20)."""
    g = _gen(seed, name)
    x = torch.randn((tokens, cols), generator=g, device="cuda")
    if tokens > 64:
        x[:, torch.randperm(cols, generator=g, device="cuda")[:max(1, cols // 100)]] *= 20
    return x.to(torch.bfloat16)


def _layer_inputs(case, seed):
    n, h = case["tokens"], case["hidden"]
    s = {"x": _activations(seed, "x", n, h), "a": _activations(seed, "a", n, case["attn"]),
         "h": torch.randn((n, h), generator=_gen(seed, "h"), device="cuda") * 4,
         "w1": torch.rand(h, generator=_gen(seed, "w1"), device="cuda") + 0.5,
         "w2": torch.rand(h, generator=_gen(seed, "w2"), device="cuda") + 0.5}
    if case["rank"]:
        r, i = case["rank"], case["inter"]
        # A of the gate and up modules stacked, and of down (whole 16-row tiles: rank 8 is padded with zero rows)
        a2 = torch.zeros((-(-r // 16) * 16, i), device="cuda")
        a2[:r] = torch.randn((r, i), generator=_gen(seed, "a2"), device="cuda") * i**-0.5
        s["la1"] = (torch.randn((2 * r, h), generator=_gen(seed, "a1"), device="cuda") * h**-0.5).to(torch.bfloat16)
        s["la2"] = a2.to(torch.bfloat16)
        s["lb1"] = (torch.randn((2 * i, r), generator=_gen(seed, "b1"), device="cuda") * 0.1).half()  # stored order
        s["lb2"] = (torch.randn((h, r), generator=_gen(seed, "b2"), device="cuda") * 0.1).half()
        s["slot"] = torch.randint(0, 3, (n,), generator=_gen(seed, "slot"), device="cuda", dtype=torch.int32)
        s["slot_scale"] = torch.tensor([0.0, 1.0, 2.0], device="cuda")  # slot 0: tokens without the adapter
    return s


def _interleave(rows):
    """The order in which [gate; up] rows are packed: tiles of 8 gate and 8 up rows."""
    half = torch.arange(rows // 2, device="cuda").reshape(-1, 8)
    return torch.cat((half, half + rows // 2), 1).reshape(-1)


def _prepare_layer(case, seed):
    n, h, inter = case["tokens"], case["hidden"], case["inter"]
    s = _layer_inputs(case, seed)
    m = _matrices(case, seed)
    s["mqkv"], s["mout"], s["mdown"] = _mat([m["qkv"]]), _mat([m["out"]]), _mat([m["down"]])
    s["mgu"] = _mat([m["gate"], m["up"]], silu=True)
    del m

    def f32(*shape):
        return torch.empty(shape, device="cuda")

    s["whole"] = n <= WHOLE_TOKENS
    s["pqkv"] = f32(1 if s["whole"] else s["mqkv"].split(n), n, case["qkv"])
    s["qkv"] = s["pqkv"][0] if s["pqkv"].shape[0] == 1 else f32(n, case["qkv"])
    s["pout"] = f32(s["mout"].split(n), n, h)
    s["pdown"] = f32(s["mdown"].split(n), n, h)
    s["y1"], s["y2"] = (torch.empty((n, h), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    s["mid"] = torch.empty((n, inter), dtype=torch.bfloat16, device="cuda")
    r = case["rank"]
    if r:
        s["mla1"], s["mla2"] = _mat([s.pop("la1")]), _mat([s.pop("la2")])
        s["xa1"] = f32(s["mla1"].split(n), n, s["mla1"].rows)
        s["xa2"] = f32(s["mla2"].split(n), n, s["mla2"].rows)
        s["lb1"] = s["lb1"][_interleave(2 * inter)].contiguous()
        s["tab1"] = torch.tensor([INT_MAX] * 4 + [0, r, -1, -1], dtype=torch.int32, device="cuda")
        s["tab2"] = torch.tensor([INT_MAX] * 4 + [0, -1, -1, -1], dtype=torch.int32, device="cuda")
    s["n"], s["rank"], s["hidden"] = n, r, h
    s["outputs"] = {"qkv": s["qkv"], "h": s["h"], "y1": s["y1"], "mid": s["mid"], "y2": s["y2"]}
    s["graph"] = _capture(lambda stream: _launch_layer(stream, s)) if n <= GRAPH_TOKENS else None
    return s


def _capture(launch):
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    return Graph.capture(stream, lambda: launch(stream))


def _launch_layer(stream, s):
    gemm, n, h = _gemm(), s["n"], s["hidden"]
    split = gemm.run_split(stream, n, s["mqkv"], s["x"], s["pqkv"], Epi.Plain, s["whole"])
    if split > 1:
        sum_parts(stream, s["pqkv"], split, n, s["mqkv"].rows, s["qkv"])
    split = gemm.run(stream, n, s["mout"], s["a"], s["pout"])
    add_rmsnorm(stream, s["h"], s["pout"], split, n, h, s["w1"], s["y1"], EPS)
    if s["rank"]:
        xs = gemm.run(stream, n, s["mla1"], s["y1"], s["xa1"])
        gemm.run_lora(stream, n, s["mgu"], s["y1"], s["mid"], Epi.Silu,
                      (s["xa1"], xs, s["mla1"].rows, s["lb1"], s["rank"], s["tab1"], s["slot"], s["slot_scale"]))
        xs = gemm.run(stream, n, s["mla2"], s["mid"], s["xa2"])
        split = gemm.run_lora(stream, n, s["mdown"], s["mid"], s["pdown"], Epi.Plain,
                              (s["xa2"], xs, s["mla2"].rows, s["lb2"], s["rank"], s["tab2"], s["slot"],
                               s["slot_scale"]))
    else:
        gemm.run(stream, n, s["mgu"], s["y1"], s["mid"], Epi.Silu)
        split = gemm.run(stream, n, s["mdown"], s["mid"], s["pdown"])
    add_rmsnorm(stream, s["h"], s["pdown"], split, n, h, s["w2"], s["y2"], EPS)


def _launch_head(stream, s):
    s["keys"].zero_()
    _gemm().run(stream, s["n"], s["mat"], s["x"], s["logits"], Epi.Argmax, n_out=s["n"], keys=s["keys"])


def _prepare_matrix(case, seed):
    what, rows, cols = case["what"], case["rows"], case["cols"]
    stored = _stored(seed, "matrix", case["weights"], rows, cols)
    if what == "dequant":
        bits, group, words, scales, zeros = stored
        return {"q": words, "scales": scales, "zeros": zeros.to(torch.uint8), "rows": rows, "words": words.shape[1],
                "cols": cols, "group": group, "bits": bits, "f32": case["f32"],
                "out": torch.empty((rows, cols), dtype=torch.float32 if case["f32"] else torch.bfloat16,
                                   device="cuda")}
    n = case["tokens"]
    s = {"n": n, "mat": _mat([stored]), "x": _activations(seed, "x", n, cols)}
    if what == "product":
        s["split"] = 1 if n <= WHOLE_TOKENS else s["mat"].split(n)
        s["parts"] = torch.empty((s["split"], n, rows), device="cuda")
        s["y"] = torch.empty((n, rows), device="cuda") if s["split"] > 1 else s["parts"][0]
        return s
    s["logits"] = torch.empty((n, rows), device="cuda")
    s["keys"] = torch.zeros(n, dtype=torch.int64, device="cuda")
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        s["graph"] = Graph.capture(stream, lambda: _launch_head(stream, s))
    return s


def prepare(case, seed):
    s = _prepare_layer(case, seed) if case["what"] == "layer" else _prepare_matrix(case, seed)
    s["what"] = case["what"]
    return s


def run(state):
    s = state
    if s["what"] == "layer":
        if s["graph"] is not None:
            s["graph"].launch(None)
        else:
            _launch_layer(None, s)
        return s["outputs"]
    if s["what"] == "head":
        s["graph"].launch(None)
        # the low half of a key is ~token
        return {"logits": s["logits"], "token": s["keys"].view(torch.int32).reshape(-1, 2)[:, 0]}
    if s["what"] == "product":
        split = _gemm().run_split(None, s["n"], s["mat"], s["x"], s["parts"], Epi.Plain, s["n"] <= WHOLE_TOKENS)
        if split > 1:
            sum_parts(None, s["parts"], split, s["n"], s["mat"].rows, s["y"])
        return s["y"]
    dequant(None, s["q"], s["scales"], s["zeros"], s["rows"], s["words"], s["cols"], s["group"], s["bits"], 0,
            s["rows"], s["out"], s["f32"])
    return s["out"]


# ---- what a pass cannot do without, and its results in 64 bits -------------------------------------------------------


def _weight_bytes(weights, rows, cols):
    """Codes, scales (bf16 values; one per 128 columns, or per row) and zero points."""
    g = rows * (cols // 128)
    return {"i4": rows * cols / 2 + 2 * g, "i4z": rows * cols / 2 + 2.5 * g, "i8g": rows * cols + 2 * g,
            "i8": rows * cols + 2 * rows, "bf16": rows * cols * 2}[weights]


def work(case):
    w = case["weights"]
    if case["what"] == "dequant":
        rows, cols = case["rows"], case["cols"]
        bits = 4 if w in ("i4", "i4z") else 8
        return {"bytes": rows * cols * bits / 8 + rows * (cols // 128) * 5 + rows * cols * (4 if case["f32"] else 2),
                "flops": 0}
    n = case["tokens"]
    if case["what"] in ("product", "head"):
        rows, cols = case["rows"], case["cols"]
        return {"bytes": _weight_bytes(w, rows, cols) + n * cols * 2 + n * rows * 4, "flops": 2 * n * rows * cols}
    h, q, a, i, r = case["hidden"], case["qkv"], case["attn"], case["inter"], case["rank"]
    shapes = [(q, h), (h, a), (2 * i, h), (h, i)]
    extra = [(2 * r, h), (2 * i, r), (r, i), (h, r)] if r else []
    # x and a in, qkv out (f32), h in and out (f32), mid and both normed rows out (bf16)
    return {"bytes": sum(_weight_bytes(w, *s) for s in shapes) + sum(2 * x * y for x, y in extra) +
            n * (2 * h + 2 * a + 4 * q + 8 * h + 2 * i + 4 * h) + 8 * h,
            "flops": 2 * n * sum(x * y for x, y in shapes + extra)}


def tolerance(case):
    if case["what"] == "dequant":
        return "exact"  # one rounding of one product per value
    n = case["tokens"]
    if case["what"] == "layer":
        # bf16 results travel through the layer: one rounding of each normed row and of the SwiGLU output
        return {"rel": 1e-2, "max": 0.3}
    if n > 32:
        return {"rel": 1e-2, "max": 0.1}  # kernels for many tokens may round each dequantized weight to 16 bits
    return {"rel": 1e-5, "max": 1e-4}  # exact products, f32 sums


def _product64(stored, x, out=None):
    """x . w^T in 64 bits, a slice of rows at a time."""
    rows = stored.shape[0] if isinstance(stored, torch.Tensor) else stored[2].shape[0]
    parts = []
    for r in range(0, rows, 16384):
        part = stored[r:r + 16384] if isinstance(stored, torch.Tensor) else \
            (*stored[:2], *(t[r:r + 16384] for t in stored[2:]))
        parts.append(x @ _dense64(part).T.contiguous())
    return torch.cat(parts, 1)


def _norm64(h, w):
    return w.double() * h / torch.sqrt((h * h).mean(1, keepdim=True) + EPS)


def exact(case, seed):
    what = case["what"]
    if what == "dequant":
        out = _dense64(_stored(seed, "matrix", case["weights"], case["rows"], case["cols"]))
        return out if case["f32"] else out.float().to(torch.bfloat16)
    if what in ("product", "head"):
        stored = _stored(seed, "matrix", case["weights"], case["rows"], case["cols"])
        y = _product64(stored, _activations(seed, "x", case["tokens"], case["cols"]).double())
        return y if what == "product" else {"logits": y, "token": None}
    s, m = _layer_inputs(case, seed), _matrices(case, seed)
    qkv = _product64(m["qkv"], s["x"].double())
    h = s["h"].double() + _product64(m["out"], s["a"].double())
    y1 = _norm64(h, s["w1"])
    gate, up = _product64(m["gate"], y1), _product64(m["up"], y1)
    r = case["rank"]
    if r:
        scale = s["slot_scale"].double()[s["slot"].long()][:, None]
        xa, i = y1 @ s["la1"].double().T.contiguous(), case["inter"]
        gate = gate + scale * (xa[:, :r] @ s["lb1"][:i].double().T.contiguous())
        up = up + scale * (xa[:, r:] @ s["lb1"][i:].double().T.contiguous())
    mid = gate * torch.sigmoid(gate) * up
    h = h + _product64(m["down"], mid)
    if r:
        h = h + scale * ((mid @ s["la2"].double().T.contiguous())[:, :r] @ s["lb2"].double().T.contiguous())
    return {"qkv": qkv, "h": h, "y1": y1, "mid": mid, "y2": _norm64(h, s["w2"])}
