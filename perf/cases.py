"""What this framework is timed on: calls of its public entry points, as a program that uses it makes them.

    listed()                 the cases
    draw(rng)                one more case of the same ranges
    prepare(case, seed)      what the program holds before the call (tensors on the GPU)
    run(state)               one pass; returns everything the pass computes
    work(case)               bytes and operations the pass cannot do without
    tolerance(case)          how far two correct implementations may be apart

Five kinds of call:

    multiply   y = M x for one vector (`multiply`; int8 values: `multiply_int8`), or with the epilogue
               y = M x + y / 2 in place (`multiply_axpby`, `multiply_int8_axpby`)
    batched    Y = X M^T for several vectors (`multiply_batched`)
    compress   dense matrix -> compressed matrix (`compress`, `compress_int8`)
    decode     one token through `DecodeEngine.step`: all projections compressed, KV cache of `context` tokens
    prefill    a prompt through `LlamaDecoder` with `MackoLinear` projections (batched products)

Matrices are N(0, 0.02) weights; "pruned" keeps the largest |w| of every row (equal rows), "bernoulli"
drops elements independently, "skewed" draws every row's density from a power law, with all-zero rows
and a 40-column gap in every row.
"""
import math

import torch

import macko_spmv_amd as mk
from macko_spmv_amd import llm

VOCAB = 32000


def listed():
    return [
        # the smallest calls: a matrix of a small model, odd sizes; launch and host path are what counts
        {"name": "multiply_small", "kind": "multiply", "rows": 777, "cols": 3333, "density": 0.25,
         "pattern": "bernoulli", "dtype": "fp16", "epilogue": False},
        # one projection of a 7B-geometry decoder at the density the format is quoted at
        {"name": "multiply_ordinary", "kind": "multiply", "rows": 11008, "cols": 4096, "density": 0.5,
         "pattern": "pruned", "dtype": "fp16", "epilogue": False},
        # ... and a wide one at the low end of the densities
        {"name": "multiply_sparse", "kind": "multiply", "rows": 4096, "cols": 11008, "density": 0.1,
         "pattern": "pruned", "dtype": "fp16", "epilogue": False},
        # the largest layers: hundreds of MB of compressed stream
        {"name": "multiply_large", "kind": "multiply", "rows": 49152, "cols": 12288, "density": 0.3,
         "pattern": "bernoulli", "dtype": "fp16", "epilogue": False},
        # rows of very uneven length, empty rows, padding entries in every row
        {"name": "multiply_skewed", "kind": "multiply", "rows": 14336, "cols": 4096, "density": 0.3,
         "pattern": "skewed", "dtype": "fp16", "epilogue": False},
        # far fewer rows than the GPU has wavefronts, long vector
        {"name": "multiply_few_rows", "kind": "multiply", "rows": 512, "cols": 16384, "density": 0.5,
         "pattern": "bernoulli", "dtype": "fp16", "epilogue": False},
        # int8 values, residual added in place
        {"name": "multiply_int8_residual", "kind": "multiply", "rows": 11008, "cols": 4096, "density": 0.5,
         "pattern": "pruned", "dtype": "int8", "epilogue": True},
        # a handful of sequences decoded together
        {"name": "batched_8", "kind": "batched", "rows": 4096, "cols": 4096, "density": 0.5,
         "pattern": "pruned", "batch": 8},
        # all tokens of a prompt through one projection
        {"name": "batched_128", "kind": "batched", "rows": 11008, "cols": 4096, "density": 0.5,
         "pattern": "pruned", "batch": 128},
        # preparing a model: one of its weight matrices
        {"name": "compress", "kind": "compress", "rows": 11008, "cols": 4096, "density": 0.5,
         "pattern": "pruned", "dtype": "fp16"},
        # generating: one token, 384 in the cache (a 128-token prompt and 256 generated)
        {"name": "decode_step", "kind": "decode", "layers": 8, "dim": 4096, "hidden": 11008, "heads": 32,
         "density": 0.5, "context": 384, "max_len": 512},
        # reading a 128-token prompt
        {"name": "prefill", "kind": "prefill", "layers": 4, "dim": 4096, "hidden": 11008, "heads": 32,
         "density": 0.5, "prompt": 128, "max_len": 512},
    ]


# ---- drawn cases ------------------------------------------------------------------------------------

def _log_int(rng, lo, hi):
    """An integer of [lo, hi], even over its logarithm; odd ones as likely as even ones."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _density(rng):
    return round(math.exp(rng.uniform(math.log(0.05), math.log(0.95))), 3)


def _size(rng, lo, hi_rows, hi_cols, most):
    """rows, cols with rows * cols <= most; half of the cols multiples of 64, as layers have."""
    while True:
        rows, cols = _log_int(rng, lo, hi_rows), _log_int(rng, 2 * lo, hi_cols)
        if rng.random() < 0.5:
            cols = max(128, cols // 64 * 64)
        if rows * cols <= most:
            return rows, cols


def draw(rng):
    kind = rng.choice(("multiply", "multiply", "multiply", "batched", "batched", "compress", "decode", "prefill"))
    if kind in ("multiply", "compress"):
        rows, cols = _size(rng, 64, 49152, 49152, 28672 * 8192 if kind == "compress" else 49152 * 12288)
        case = {"kind": kind, "rows": rows, "cols": cols, "density": _density(rng),
                "pattern": rng.choice(("pruned", "bernoulli", "bernoulli", "skewed")),
                "dtype": rng.choice(("fp16", "fp16", "int8"))}
        if case["pattern"] == "skewed":
            case["density"] = 0.3
        if kind == "multiply":
            case["epilogue"] = rng.random() < 0.3
            # no more stored entries than the largest listed matrix has
            case["density"] = min(case["density"], round(0.3 * 49152 * 12288 / (rows * cols), 3))
        return case
    if kind == "batched":
        while True:
            rows, cols = _size(rng, 64, 28672, 28672, 11008 * 11008)
            batch, density = _log_int(rng, 2, 256), _density(rng)
            if rows * cols * batch * density <= 11008 * 4096 * 128:
                return {"kind": kind, "rows": rows, "cols": cols, "density": density,
                        "pattern": rng.choice(("pruned", "bernoulli")), "batch": batch}
    dim, hidden, heads = rng.choice(((512, 1376, 8), (1024, 2752, 8), (2048, 5504, 16), (4096, 11008, 32)))
    case = {"kind": kind, "dim": dim, "hidden": hidden, "heads": heads, "density": _density(rng)}
    if kind == "decode":
        case["layers"] = rng.randint(1, 8)
        case["context"] = _log_int(rng, 1, 2047)
        case["max_len"] = (case["context"] + 512) // 512 * 512
    else:
        case["layers"] = rng.randint(1, 4)
        case["prompt"] = _log_int(rng, 2, 128)
        case["max_len"] = 512
    return case


# ---- inputs -----------------------------------------------------------------------------------------

def _skewed_densities(rows, mean, uniform):
    """Power-law row densities (alpha 1.5) clipped to [0.01, 0.95] and rescaled to the wanted mean."""
    d = (0.01 * (1.0 - uniform) ** (-1.0 / 1.5)).clamp(0.01, 0.95)
    for _ in range(20):
        d = (d * (mean / d.mean())).clamp(0.01, 0.95)
    return d


def _matrix(case, generator):
    rows, cols, density = case["rows"], case["cols"], case["density"]
    w = torch.randn((rows, cols), device="cuda", generator=generator, dtype=torch.float16).mul_(0.02)
    if case["pattern"] == "pruned":
        llm.prune_rows_(w, density)
    else:
        if case["pattern"] == "skewed":
            u = torch.rand((rows,), device="cuda", generator=generator)
            density = _skewed_densities(rows, density, u)[:, None]
        w.mul_(torch.rand((rows, cols), device="cuda", generator=generator) < density)
        if case["pattern"] == "skewed":
            gap = min(40, cols // 4)
            start = torch.randint(0, cols - gap, (rows, 1), device="cuda", generator=generator)
            column = torch.arange(cols, device="cuda")[None, :]
            w.masked_fill_((column >= start) & (column < start + gap), 0)
            w[::97] = 0
    if case.get("dtype") == "int8":
        # symmetric quantisation; an element that survived the pruning stays non-zero
        q = torch.clamp(torch.round(w.float() * (127.0 / 0.08)), -127, 127).to(torch.int8)
        return torch.where((q == 0) & (w != 0), torch.ones_like(q), q).contiguous()
    return w.contiguous()


def _vectors(shape, generator):
    return torch.randn(shape, device="cuda", generator=generator, dtype=torch.float16)


def _model(case, seed):
    """Decoder of the case's geometry, random weights, every projection pruned and compressed."""
    torch.manual_seed(seed)
    with torch.device("cuda"):
        model = llm.LlamaDecoder(VOCAB, case["dim"], case["hidden"], case["layers"], case["heads"], case["max_len"])
    model = model.half().requires_grad_(False)
    for layer in model.model.layers:
        for parent, name in llm.PROJECTIONS:
            module = getattr(layer, parent)
            w = getattr(module, name).weight.data.normal_(0.0, 0.02)
            llm.prune_rows_(w, case["density"])
            setattr(module, name, llm.MackoLinear(*mk.compress(w)))
    return model


def prepare(case, seed):
    kind = case["kind"]
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed)
    if kind == "decode":
        engine = llm.DecodeEngine(_model(case, seed))
        for entry in engine.layers:
            for key in ("k_cache", "v_cache"):
                entry[key][:, :case["context"]] = _vectors((case["heads"], case["context"], case["dim"] // case["heads"]),
                                                           generator)
        token = torch.randint(0, VOCAB, (1,), device="cuda", generator=generator)
        return {"kind": kind, "engine": engine, "token": token,
                "position": torch.tensor([case["context"]], device="cuda")}
    if kind == "prefill":
        model = _model(case, seed)
        return {"kind": kind, "model": model,
                "tokens": torch.randint(0, VOCAB, (1, case["prompt"]), device="cuda", generator=generator),
                "positions": torch.arange(case["prompt"], device="cuda")}
    int8 = case.get("dtype") == "int8"
    if kind == "compress":
        # one matrix per case, its rows in an order of the seed's: the lengths of the outputs depend on
        # the number of zeros in every gap, and are the same for every order of the rows
        matrix = _matrix(case, torch.Generator(device="cuda").manual_seed(20))
        order = torch.randperm(case["rows"], device="cuda", generator=generator)
        return {"kind": kind, "int8": int8, "matrix": matrix.index_select(0, order)}
    matrix = _matrix(case, generator)
    state = {"kind": kind, "int8": int8, "compressed": mk.compress_int8(matrix) if int8 else mk.compress(matrix)}
    del matrix
    if kind == "batched":
        state["x"] = _vectors((case["batch"], case["cols"]), generator)
    else:
        state["x"] = _vectors((case["cols"],), generator)
        state["y"] = _vectors((case["rows"],), generator) if case["epilogue"] else None
    return state


def run(state):
    kind = state["kind"]
    if kind == "multiply":
        if state["y"] is not None:
            product = mk.multiply_int8_axpby if state["int8"] else mk.multiply_axpby
            return product(state["compressed"], state["x"], state["y"], 1.0, 0.5)
        return (mk.multiply_int8 if state["int8"] else mk.multiply)(state["compressed"], state["x"])
    if kind == "batched":
        return mk.multiply_batched(state["compressed"], state["x"])
    if kind == "compress":
        return (mk.compress_int8 if state["int8"] else mk.compress)(state["matrix"])
    if kind == "decode":
        engine = state["engine"]
        logits = engine.step(state["token"], state["position"])
        return [logits, [(entry["k_cache"], entry["v_cache"]) for entry in engine.layers]]
    model = state["model"]
    logits = model(state["tokens"], state["positions"])
    return [logits, [(layer.self_attn.k_cache, layer.self_attn.v_cache) for layer in model.model.layers]]


# ---- what a pass cannot do without ------------------------------------------------------------------

def _entries(rows, cols, density, pattern="pruned"):
    """Expected stored entries: the non-zeros, and one padding entry per 16 zeros of a gap."""
    if pattern == "skewed":
        u = (torch.arange(2048, dtype=torch.float64) + 0.5) / 2048
        d = _skewed_densities(2048, density, u)
        per_row = float((d * cols / (1.0 - (1.0 - d) ** 16)).mean())
        return rows * per_row * (96 / 97)
    kept = round(density * cols) if pattern == "pruned" else density * cols
    return rows * kept / max(1e-9, 1.0 - (1.0 - density) ** 16)


def _compressed_bytes(rows, entries, value_bytes=2):
    return entries * (value_bytes + 0.5) + 4 * (rows + 1)


def work(case):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        dim, hidden, layers, density = case["dim"], case["hidden"], case["layers"], case["density"]
        tokens = case.get("prompt", 1)
        rows = 5 * dim + 2 * hidden  # q, k, v, o and down: dim each; gate, up: hidden each
        entries = _entries(4 * dim + 2 * hidden, dim, density) + _entries(dim, hidden, density)
        weights = layers * _compressed_bytes(rows, entries)
        # keys and values: the cached ones read, the new ones written
        cached = case.get("context", tokens)
        cache = layers * 2 * 2 * dim * (cached + tokens)
        head = 2 * VOCAB * dim
        pairs = tokens * cached if kind == "decode" else tokens * (tokens + 1) / 2
        return {"bytes": weights + cache + head + 2 * tokens * (VOCAB + dim),
                "flops": 2 * tokens * (layers * entries + VOCAB * dim) + layers * 4 * dim * pairs}
    rows, cols = case["rows"], case["cols"]
    value_bytes = 1 if case.get("dtype") == "int8" else 2
    entries = _entries(rows, cols, case["density"], case["pattern"])
    stored = _compressed_bytes(rows, entries, value_bytes)
    if kind == "compress":
        return {"bytes": value_bytes * rows * cols + stored, "flops": 0}
    batch = case.get("batch", 1)
    vectors = 2 * batch * (cols + rows) + (2 * rows if case.get("epilogue") else 0)
    return {"bytes": stored + vectors, "flops": 2 * entries * batch}


def tolerance(case):
    kind = case["kind"]
    if kind == "compress":
        return "exact"
    if kind in ("decode", "prefill"):
        # fp16 activations between the layers: a sum in another order moves some of them by one unit in
        # the last place, and the layers behind carry that on.  Against the same model in float64:
        # rel 1.9e-3, largest 1.6e-2 (keys and values of the last layer of a prompt); four times that.
        return {"rel": 7.5e-3, "max": 0.066}
    # fp32 sums rounded once to fp16.  Against float64 products: rel 2.1e-4, largest 4.9e-4 (half a unit
    # in the last place) for every matrix here; four times that.
    return {"rel": 8.4e-4, "max": 2e-3}
