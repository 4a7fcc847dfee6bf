"""The work whose speed is watched: what an inference worker has this package do on one GPU.

Six kinds of work, each through the package's public functions as a worker calls them:

bulk      an engine step's SwiftKV write: the K/V of every skipped layer scattered into the paged caches by
          slot_mapping (eager, as the step is), and in a step that ends prompts also the selection of the rows that go
          on to the decode runner
decode    one decode step as a captured HIP graph: the bulk write, ln0, three LSTM speculator steps
lstm      the LSTM speculator's proposal round without its matrix products: ln0 / sqrt 2, then per head the gate update
          from the looked-up embedding and the token selection; a captured HIP graph per padded batch size
gates     the same operators as the speculator issues them without the embedding lookup folded in: eager, pre-activations
          of both projections given
mlp       the MLP speculator's proposal round, eager: ln0 / sqrt 2, then per head embedding + add + norm + GELU and the
          token selection
fp4       one layer's NVFP4-style cache write

The matrix products between these steps belong to the model; their outputs (projections, logits) are inputs here.
"""
import math

import torch

import arcticinference_amd as ops

DEVICE = "cuda:0"
BLOCK_SIZE = 16
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
WIDTHS = [1024, 2048, 2880, 3072, 4000, 4096, 5120, 6144, 8192]
VOCABULARIES = [32000, 50257, 65536, 128256, 128257, 151936]


def _bulk(name, tokens, layers, heads, head_size, dtype="bf16", cache="fp8", blocks=0, padding=0.0, std=1.5, selected=0,
          hidden=0):
    case = {"kind": "bulk", "tokens": tokens, "layers": layers, "heads": heads, "head_size": head_size, "dtype": dtype,
            "cache": cache, "blocks": blocks or 2 * -(-tokens // BLOCK_SIZE) + 8, "padding": padding, "std": std,
            "selected": selected, "hidden": hidden}
    return dict(case, name=name) if name else case


def _spec(name, kind, rows, width, vocabulary, dtype="bf16", heads=3, pad=0, affine=True, fast_gelu=False):
    case = {"kind": kind, "rows": rows, "width": width, "vocabulary": vocabulary, "dtype": dtype, "heads": heads, "pad": pad,
            "affine": affine, "fast_gelu": fast_gelu}
    return dict(case, name=name) if name else case


def listed():
    return [
        # the prefill chunk of a 70B SwiftKV model (80 layers, the upper 40 skipped), 10 % padding: the benchmark's headline
        _bulk("prefill_70b_fp8", 16384, 40, 8, 128, blocks=8192, padding=0.10),
        # the prefill chunk of an 8B SwiftKV model (32 layers, the upper 16 skipped)
        _bulk("prefill_8b_fp8", 8192, 16, 8, 128, blocks=8192),
        # a mixed step of the 70B model: part of a prompt among decodes, no round number of tokens, and the selection of
        # the 61 rows that continue (K/V with the write; hidden states, residual and positions beside it)
        _bulk("mixed_step_70b_select", 2173, 40, 8, 128, selected=61, hidden=8192),
        # a step of decodes with an unquantised cache
        _bulk("decode_8b_bf16_cache", 256, 16, 8, 128, cache="auto", blocks=512, std=1.0),
        # the smallest step: a handful of requests decode
        _bulk("decode_few_8b_fp8", 5, 16, 8, 128),
        # a chunk of a model whose rows are no power of two long and whose activations are fp16
        _bulk("prefill_ragged_rows_fp16", 5003, 33, 3, 96, dtype="fp16", padding=0.05),
        # the decode step of 512 requests at the 8B shape as one graph
        {"name": "decode_step_graph", "kind": "decode", "tokens": 512, "layers": 16, "heads": 8, "head_size": 128, "blocks": 32768,
         "width": 4096, "dtype": "bf16"},
        # a proposal round for a full batch and for a few requests
        _spec("lstm_round_512", "lstm", 512, 4096, 128256),
        _spec("lstm_round_7", "lstm", 7, 4096, 128256),
        # the MLP speculator's round for a middling batch, an odd vocabulary (every row of logits starts elsewhere)
        _spec("mlp_round_64_fp16", "mlp", 64, 2880, 50257, dtype="fp16"),
        # widths and pitches that no vector access fits, as the operators' unit tests have them; the norms without scale and shift
        _spec("gates_odd_width_fp16", "gates", 300, 1537, 0, dtype="fp16", pad=3, affine=False),
        # one layer's fp4 write of a prefill chunk
        {"name": "fp4_layer_8192", "kind": "fp4", "tokens": 8192, "heads": 8, "head_size": 128, "dtype": "bf16", "heads_first": False},
    ]


def _between(rng, low, high):
    """A size from the whole range, spread over its logarithm, odd ones among them."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(["bulk", "bulk", "bulk", "decode", "lstm", "lstm", "mlp", "gates", "gates", "fp4"])
    if kind == "bulk":
        layers = rng.choice([1, 8, 16, 16, 33, 40, 40])
        heads, head_size = rng.choice([(8, 128)] * 4 + [(1, 128), (2, 128), (4, 128), (8, 64), (3, 96), (3, 80)])
        tokens = _between(rng, 1, 16384)
        case = _bulk(None, tokens, layers, heads, head_size, dtype=rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"]),
                     cache=rng.choice(["fp8", "fp8", "fp8_e5m2", "auto"]), padding=rng.choice([0.0, 0.0, 0.1, 0.3]),
                     selected=rng.choice([0, 0, _between(rng, 1, min(tokens, 512))]), hidden=rng.choice([4096, 8192]))
        most = work(_bulk(None, 16384, 40, 8, 128, padding=0.1))["bytes"]
        while work(case)["bytes"] > most:   # fp32 sources and unquantised caches move more per token
            case["tokens"] //= 2
            case["selected"] = min(case["selected"], case["tokens"])
        return case
    if kind == "decode":
        return {"kind": "decode", "tokens": _between(rng, 1, 512), "layers": rng.choice([16, 40]), "heads": 8, "head_size": 128,
                "blocks": 4096, "width": rng.choice(WIDTHS), "dtype": rng.choice(["bf16", "fp16"])}
    if kind == "fp4":
        heads, head_size = rng.choice([(8, 128), (8, 128), (1, 128), (2, 64), (3, 80)])
        return {"kind": "fp4", "tokens": _between(rng, 1, 32768), "heads": heads, "head_size": head_size,
                "dtype": rng.choice(["bf16", "fp16"]), "heads_first": rng.random() < 0.5}
    if kind == "gates":
        return _spec(None, kind, _between(rng, 1, 4096), rng.choice([rng.choice(WIDTHS), rng.choice(WIDTHS), _between(rng, 64, 8200)]), 0,
                     dtype=rng.choice(["bf16", "fp16"]), pad=rng.choice([0, 0, 8, 3]), affine=rng.random() < 0.7,
                     fast_gelu=rng.random() < 0.2)
    return _spec(None, kind, _between(rng, 1, 512), rng.choice(WIDTHS), rng.choice(VOCABULARIES), dtype=rng.choice(["bf16", "fp16"]))


# --- what a worker has in hand before the call ------------------------------------------------------------------------

class State:
    """The tensors of one case and, where the worker replays a graph, the graph with its outputs."""

    def __init__(self, case, seed):
        self.case = case
        self.generator = torch.Generator(device=DEVICE).manual_seed(seed)
        self.dtype = DTYPES[case["dtype"]]
        self.graph = None

    def normal(self, *shape, std=1.0, mean=0.0, dtype=None):
        x = torch.empty(shape, dtype=dtype or self.dtype, device=DEVICE)
        return x.normal_(mean, std, generator=self.generator)

    def below(self, limit, *shape):
        return torch.randint(0, limit, shape, generator=self.generator, device=DEVICE)

    def capture(self, step):
        step()
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.outputs = step()


def _prepare_kv(s, cache, std):
    c = s.case
    n = c["heads"] * c["head_size"]
    s.keys = s.normal(c["tokens"], c["layers"] * n, std=std)
    s.values = s.normal(c["tokens"], c["layers"] * n, std=std)
    s.slots = torch.randperm(c["blocks"] * BLOCK_SIZE, generator=s.generator, device=DEVICE)[:c["tokens"]].contiguous()
    if c.get("padding"):
        s.slots[torch.rand(c["tokens"], generator=s.generator, device=DEVICE) < c["padding"]] = -1
    element = s.dtype if cache == "auto" else torch.uint8
    s.pools = [torch.empty(2, c["blocks"], BLOCK_SIZE, c["heads"], c["head_size"], dtype=element, device=DEVICE).fill_(layer + 1)
               for layer in range(c["layers"])]
    largest = 57344.0 if cache == "fp8_e5m2" else 448.0
    scale = [(x.view(c["tokens"], c["layers"], n).abs().amax(dim=(0, 2)).float() / largest).unbind() for x in (s.keys, s.values)]
    s.layers = ([p[0] for p in s.pools], [p[1] for p in s.pools])
    s.scales = ([v.clone() for v in scale[0]], [v.clone() for v in scale[1]])


def _write(s, cache):
    ops.reshape_and_cache_flash_bulk(s.keys, s.values, *s.layers, s.slots, cache, *s.scales, s.case["heads"], s.case["head_size"])


def _prepare_gate_vectors(s, width, affine=True):
    s.vectors = [s.normal(width, std=0.02, mean=mean) if affine else None for mean in (1.0, 0.0, 1.0, 0.0)]
    state_weight = 0.5 ** (0.5 / 3)
    s.alpha = math.sqrt((1 - state_weight * state_weight) * (width / 2)) / state_weight


def _pitched(s, rows, width, pad, gates=1):
    return s.normal(rows, gates * width + pad)[:, :gates * width]


def prepare(case, seed):
    if not ops.try_load_torch_library():
        raise RuntimeError("the operators are not built")
    s = State(case, seed)
    kind = case["kind"]
    if kind == "bulk":
        _prepare_kv(s, case["cache"], case["std"])
        if case["selected"]:
            tokens, width = s.keys.shape
            s.rows = [s.normal(tokens, case["hidden"]), s.normal(tokens, case["hidden"]), s.below(1 << 17, tokens)]
            s.indices = torch.randperm(tokens, generator=s.generator, device=DEVICE)[:case["selected"]].sort().values
            made = lambda like, *shape: torch.zeros(case["selected"], *shape, dtype=like.dtype, device=DEVICE)
            s.chosen_kv = [made(s.keys, width), made(s.values, width)]
            s.chosen = [made(r, *r.shape[1:]) for r in s.rows]
    elif kind == "decode":
        _prepare_kv(s, "fp8", 1.5)
        rows, width = case["tokens"], case["width"]
        _prepare_gate_vectors(s, width)
        s.hidden = s.normal(rows, width)
        s.projected = [s.normal(rows, 4 * width) for _ in range(3)]
        s.embedded = [s.normal(rows, width).repeat(1, 4) for _ in range(3)]

        def step():
            _write(s, "fp8")
            out = [ops.speculator_ln(s.hidden, None, None, 1e-6)]
            cell = None
            for projected, embedded in zip(s.projected, s.embedded):
                state, cell = ops.sum_lstm(projected, embedded, cell, *s.vectors, s.alpha, 1e-6, 1e-6, False)
                out += [state, cell]
            return out

        s.capture(step)
    elif kind == "fp4":
        tokens, heads, head_size = case["tokens"], case["heads"], case["head_size"]
        s.keys, s.values = s.normal(tokens, heads, head_size, std=1.5), s.normal(tokens, heads, head_size, std=1.5)
        blocks = 2 * -(-tokens // BLOCK_SIZE) + 8
        inner = (heads, BLOCK_SIZE) if case["heads_first"] else (BLOCK_SIZE, heads)
        s.cache = [torch.full((blocks, *inner, head_size // per), 7, dtype=torch.uint8, device=DEVICE) for per in (2, 2, 16, 16)]
        s.slots = torch.randperm(blocks * BLOCK_SIZE, generator=s.generator, device=DEVICE)[:tokens].contiguous()
        s.one = torch.ones((), device=DEVICE)
    else:
        rows, width, heads, vocabulary = case["rows"], case["width"], case["heads"], case["vocabulary"]
        _prepare_gate_vectors(s, width, case["affine"])
        s.hidden = _pitched(s, rows, width, case["pad"])
        gates = 1 if kind == "mlp" else 4
        s.projected = [_pitched(s, rows, width, case["pad"], gates) for _ in range(heads)]
        if kind == "gates":
            s.embedded = [_pitched(s, rows, width, case["pad"], 4) for _ in range(heads)]
            s.cell = _pitched(s, rows, width, case["pad"])
        else:
            s.table = s.normal(vocabulary, width)
            s.logits = [s.normal(rows, vocabulary, std=2.0) for _ in range(heads)]
            s.tokens = s.below(vocabulary, rows)
        if kind == "lstm":
            s.capture(lambda: _lstm_round(s))
    return s


# --- one pass ---------------------------------------------------------------------------------------------------------

def _lstm_round(s):
    out = [ops.speculator_ln_scaled(s.hidden, None, None, 1e-6, 0.5 ** 0.5)]
    tokens, cell = s.tokens, None
    for projected, logits in zip(s.projected, s.logits):
        state, cell = ops.sum_lstm_embedded(projected, s.table, tokens, cell, *s.vectors, s.alpha, 1e-6, 1e-6, False)
        tokens = ops.speculator_argmax(logits, s.case["vocabulary"])
        out += [state, cell, tokens]
    return out


def run(state):
    s, case = state, state.case
    kind = case["kind"]
    if kind == "bulk":
        if not case["selected"]:
            _write(s, case["cache"])
            return s.pools
        ops.reshape_and_cache_flash_bulk_select(s.keys, s.values, *s.layers, s.slots, case["cache"], *s.scales, case["heads"],
                                                case["head_size"], s.indices, *s.chosen_kv)
        ops.gather_rows(s.rows, s.indices, s.chosen)
        return [s.pools, s.chosen_kv, s.chosen]
    if kind == "decode":
        s.graph.replay()
        return [s.pools, s.outputs]
    if kind == "lstm":
        s.graph.replay()
        return s.outputs
    if kind == "fp4":
        ops.reshape_and_cache_flash_fp4(s.keys, s.values, s.cache[0], s.cache[1], s.cache[2], s.cache[3], s.slots, "fp4", s.one, s.one)
        return s.cache
    out = [ops.speculator_ln_scaled(s.hidden, None, None, 1e-6, 0.5 ** 0.5)]
    if kind == "mlp":
        tokens = s.tokens
        for projected, logits in zip(s.projected, s.logits):
            state = ops.speculator_embed_add_ln_gelu(projected, s.table, tokens, s.vectors[0], s.vectors[1], s.alpha, 1e-6)
            tokens = ops.speculator_argmax(logits, case["vocabulary"])
            out += [state, tokens]
        return out
    cell = s.cell
    for projected, embedded in zip(s.projected, s.embedded):
        state, cell = ops.sum_lstm(projected, embedded, cell, *s.vectors, s.alpha, 1e-6, 1e-6, case["fast_gelu"])
        out += [state, cell]
    return out


# --- what a pass cannot do without ------------------------------------------------------------------------------------

def work(case):
    """Every input read once and every output written once; arithmetic counted per element (a handful for a conversion
    or a norm, about 60 for the gate update)."""
    kind = case["kind"]
    size = DTYPES[case["dtype"]].itemsize
    if kind in ("bulk", "decode"):
        tokens, row = case["tokens"], case["layers"] * case["heads"] * case["head_size"]
        cache = case.get("cache", "fp8")
        valid = tokens * (1 - case.get("padding", 0.0))
        wide = 2 * row * size   # a token's K and V
        total = valid * (wide + (wide if cache == "auto" else 2 * row)) + 8 * tokens
        flops = 0 if cache == "auto" else 4 * valid * row
        if case.get("selected"):   # the selected rows are written again; the step's other tensors are read and written
            total += case["selected"] * (wide + 8 + 2 * (2 * case["hidden"] * size + 8))
        if kind == "decode":   # ln0, three gate updates of which the first has no previous cell
            elements = tokens * case["width"]
            total += elements * size * (2 + 10 + 11 + 11) + 4 * case["width"] * size
            flops += elements * (5 + 3 * 60)
        return {"bytes": int(total), "flops": int(flops)}
    if kind == "fp4":
        elements = 2 * case["tokens"] * case["heads"] * case["head_size"]
        return {"bytes": int(elements * (size + 0.5 + 1 / 16) + 8 * case["tokens"]), "flops": int(3 * elements)}
    rows, heads = case["rows"], case["heads"]
    elements = rows * case["width"]
    total, flops = 2 * elements * size, 5 * elements
    per_element = {"lstm": 4 + 1 + 1 + 2, "mlp": 1 + 1 + 1, "gates": 4 + 4 + 1 + 2}[kind]
    total += heads * elements * size * per_element
    flops += heads * elements * (25 if kind == "mlp" else 60)
    if kind == "lstm":
        total -= elements * size   # the first head has no previous cell
    if kind != "gates":
        total += heads * rows * (case["vocabulary"] * size + 8 + 8)
        flops += heads * rows * case["vocabulary"]
    if case["affine"]:
        total += (2 if kind == "mlp" else 4) * case["width"] * size
    return {"bytes": int(total), "flops": int(flops)}


def tolerance(case):
    """Cache bytes, selected rows and tokens are the same whatever computes them.  The speculator's outputs are rounded to
    16 bits from fp32 arithmetic whose order is free: against the same formulas in 64 bits, with the roundings to 16 bits
    where the operators have them, fourteen cases of all kinds were within 4.6e-5 (and 1.4e-2 at the worst element, a
    16-bit step of a cell that two further gate updates carry on); four times that is allowed."""
    if case["kind"] in ("bulk", "fp4"):
        return "exact"
    return {"rel": 2e-4, "max": 6e-2}
