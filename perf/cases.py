"""Performance cases of the multi-adapter LoRA path: what one forward step of a serving loop asks of this package.

A pass is one step over `layers` decoder layers: the batch's routing tables (AdapterBatchData.from_meta, once per step,
as in the reference's generate_token) and, layer by layer, the LoRA update of every projection group through the
LoRA linear layers - or the drop-in functions and the stacked-weight wrapper, for programs that call those.  The
linear layers' base product is not part of this package: base_layer hands over the buffer that holds it, and
every pass adds its update to that buffer, which is the pass's output.  Decode steps that a server would replay from a
captured graph (`graph`) keep their tables, as utils/graph.py of the reference does, and replay.

A case:
  kind      "layers": LoRA linear layers over batch tables; "dropin": lora_a_/lora_b_sgmv_cutlass and add_lora_a_/
            add_lora_b_bgmv with the reference's weight layouts, one projection at a time; "stacked": preloaded adapters
            through PunicaWrapper
  block     the projections of a layer (BLOCKS); head: width of an LM head with LoRA after the last layer, 0 = none
  dtype, layers, adapters (resident), ranks (the adapters take them in turn)
  tokens    decode rows, each of a request of its own; popularity of their adapters "uniform" or "zipf"; `bare` is the
            share of requests without adapter
  runs      prefilling requests of shortest..longest tokens (log-uniform); 0 = a decode batch
  graph     replayed from a captured graph
  route     number that the batch's adapters and lengths are drawn from; the order of the requests comes from the seed
"""

import math
import random

import torch

from lorax_amd import sgmv
from lorax_amd.adapters import (LORA, AdapterBatchData, LayerAdapterWeights, LoraConfig, LoraWeights,
                                stack_preloaded_adapters)
from lorax_amd.layers import MultiAdapterHead, TensorParallelAdapterRowLinear, TensorParallelMultiAdapterLinear
from lorax_amd.punica_wrapper import PunicaWrapper
from lorax_amd.synthetic import GQA_ATTN, LLAMA70B_LAYER, MISTRAL_MLP, ProjectionGroup, make_meta

# hidden sizes of the reference's shape table that no power of two divides: 2752 and 6848 are not multiples of 128
ODD_MLP = [ProjectionGroup("in_proj", ["in_proj"], 2752, [6848]), ProjectionGroup("out_proj", ["out_proj"], 6848, [2752])]
BLOCKS = {
    "mistral7b": GQA_ATTN + MISTRAL_MLP,
    "attention": GQA_ATTN,
    "mlp": MISTRAL_MLP,
    "llama70b": LLAMA70B_LAYER,
    "odd": ODD_MLP,
}
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
BASE_MODEL = 0  # adapter index of a request without adapter; adapters are numbered from 1
PLAIN = {"kind": "layers", "dtype": "bf16", "tokens": 0, "popularity": "uniform", "bare": 0.0, "runs": 0, "shortest": 0,
         "longest": 0, "graph": False, "head": 0}


def listed():
    def case(name, **kw):
        return {"name": name, **PLAIN, **kw}

    return [
        # One request being answered, one adapter on every projection: the smallest step there is, all latency.
        case("decode_one_request", block="mistral7b", layers=8, adapters=1, ranks="16", tokens=1, route=1),
        # A few dozen chats over a dozen adapters of different ranks, a share of them on the base model; fp16 and an
        # adapter on the LM head.
        case("decode_chat", block="mistral7b", layers=8, adapters=12, ranks="8,16,32,64", tokens=45, bare=0.1, dtype="fp16",
             head=32000, route=2),
        # The benchmark's decode batch: 256 requests over 128 rank-8 adapters on the attention projections, replayed.
        case("decode_attention_graph", block="attention", layers=16, adapters=128, ranks="8", tokens=256, bare=0.05,
             graph=True, route=3),
        # A full decode batch over hundreds of adapters with a popular few, four ranks, all projections, replayed.
        case("decode_zipf_graph", block="mistral7b", layers=2, adapters=500, ranks="8,16,32,64", tokens=512,
             popularity="zipf", graph=True, route=4),
        # Decode at the largest rank and width: all bytes.
        case("decode_70b_graph", block="llama70b", layers=1, adapters=256, ranks="128", tokens=260, bare=0.02, graph=True,
             route=5),
        # Preloaded adapters in stacked weights (PunicaWrapper), decode.
        case("decode_stacked", kind="stacked", block="mistral7b", layers=8, adapters=16, ranks="16", tokens=96, bare=0.05,
             route=6),
        # The first step of one request of ordinary length.
        case("prefill_one_request", block="mistral7b", layers=8, adapters=1, ranks="16", runs=1, shortest=300,
             longest=420, dtype="fp16", route=7),
        # Several waiting requests admitted together, about a thousand rows.
        case("prefill_thousand_rows", block="mistral7b", layers=4, adapters=10, ranks="64", runs=10, shortest=32,
             longest=256, route=8),
        # Requests whose adapters differ in rank, next to the decode rows of running ones.
        case("prefill_mixed_ranks", block="mistral7b", layers=2, adapters=24, ranks="8,16,32,64", tokens=24, runs=12,
             shortest=20, longest=900, route=9),
        # The benchmark's large prefill: 32 requests of 16 to 2048 tokens, one rank-64 adapter each, MLP.
        case("prefill_mlp_large", block="mlp", layers=1, adapters=32, ranks="64", runs=32, shortest=16, longest=2048,
             route=10),
        # A chunk of a long prompt next to 256 decode rows at the largest rank and width.
        case("mixed_70b", block="llama70b", layers=1, adapters=256, ranks="128", tokens=260, bare=0.02, runs=1,
             shortest=4096, longest=4096, route=11),
        # A program that swaps only the kernel module in: the reference's layouts, calls and zero-fills.
        case("dropin_prefill", kind="dropin", block="mistral7b", layers=1, adapters=8, ranks="32", runs=8, shortest=40,
             longest=700, route=12),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case of these ranges: any kind, block, type and set of ranks; sizes over their logarithm."""
    most = max(work(c)["bytes"] for c in listed())
    while True:
        shape = rng.choice(["decode", "decode", "graph", "graph", "stacked", "dropin decode", "prefill", "prefill", "prefill",
                            "mixed", "dropin prefill"])
        block = rng.choice(["mistral7b", "mistral7b", "attention", "mlp", "llama70b", "odd"])
        ranks = rng.choice(["8", "16", "32", "64", "128", "8,16", "16,64", "8,16,32,64"])
        case = {**PLAIN, "block": block, "dtype": rng.choice(["bf16", "bf16", "fp16"]), "ranks": ranks,
                "route": rng.randrange(1 << 20), "layers": rng.choice([1, 2, 3, 4, 6, 8])}
        if shape in ("prefill", "mixed", "dropin prefill"):
            case["runs"] = _log_uniform(rng, 1, 40)
            case["shortest"] = _log_uniform(rng, 8, 300)
            case["longest"] = _log_uniform(rng, case["shortest"], 4096)
            case["adapters"] = _log_uniform(rng, 1, 64)
            if shape == "mixed":
                case["tokens"] = _log_uniform(rng, 1, 256)
        else:
            case["tokens"] = _log_uniform(rng, 1, 512)
            case["adapters"] = _log_uniform(rng, 1, 300)
            if shape in ("decode", "graph"):
                case["head"] = rng.choice([0, 0, 0, 32000])
        case["popularity"] = rng.choice(["uniform", "zipf"])
        case["bare"] = rng.choice([0.0, 0.0, 0.05, 0.3])
        case["graph"] = shape == "graph"
        case["kind"] = "dropin" if shape.startswith("dropin") else "stacked" if shape == "stacked" else "layers"
        if case["kind"] == "stacked":
            case["ranks"] = ranks.split(",")[-1]  # a stack has one rank
            case["adapters"] = min(case["adapters"], 64)
        copies = case["adapters"] * case["layers"] * sum(len(g.layer_names) for g in BLOCKS[block])
        resident = sum((g.h_in * len(g.sizes) + g.h_out) for g in BLOCKS[block]) * case["layers"] * 2 * sum(_ranks(case).values())
        rows = sum(n for _, n in _requests(case))
        if rows <= 16384 and copies <= 14000 and resident <= 12e9 and work(case)["bytes"] <= most and _routed(case):
            return case


def _ranks(case):
    """Rank of every resident adapter."""
    ranks = [int(r) for r in case["ranks"].split(",")]
    return {a: ranks[a % len(ranks)] for a in range(1, case["adapters"] + 1)}


def _requests(case):
    """(adapter, rows) of every request of the batch."""
    rng = random.Random(case["route"])
    adapters = list(range(1, case["adapters"] + 1))
    weights = [1.0 / a**1.1 if case["popularity"] == "zipf" else 1.0 for a in adapters]
    out = []
    for i in range(case["runs"]):
        rows = _log_uniform(rng, case["shortest"], case["longest"])
        out.append((adapters[i % len(adapters)] if rng.random() >= case["bare"] else BASE_MODEL, rows))
    for a in rng.choices(adapters, weights, k=case["tokens"]):
        out.append((a if rng.random() >= case["bare"] else BASE_MODEL, 1))
    return out


def _routed(case):
    """Rows of every adapter of the batch."""
    rows = {}
    for a, n in _requests(case):
        if a != BASE_MODEL:
            rows[a] = rows.get(a, 0) + n
    return rows


class _Batch:
    """One batch in front of its forward step."""


def _randn(gen, shape, std, dtype):
    return torch.randn(shape, generator=gen, dtype=torch.float32, device="cuda").mul_(std).to(dtype)


def _adapters(case, gen, group, h_out, layers):
    layer = LayerAdapterWeights()
    dtype = DTYPES[case["dtype"]]
    for a, r in _ranks(case).items():
        wa = _randn(gen, (layers, group.h_in, r), 0.02, dtype)
        wb = _randn(gen, (layers, r, h_out), 0.02, dtype)
        layer.add_adapter(a, LoraWeights(list(wa.unbind(0)), list(wb.unbind(0)), LoraConfig(r=r)))
    return layer


def _base(y):
    """The base linear layer: its product is already in `y`."""
    return lambda x: y


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, layers = DTYPES[case["dtype"]], case["layers"]
    requests = _requests(case)
    # prefilling requests come first, each group in an order of the seed's
    order = random.Random(seed)
    runs, decode = requests[: case["runs"]], requests[case["runs"] :]
    order.shuffle(runs)
    order.shuffle(decode)
    indices = [a for a, n in runs + decode for _ in range(n)]
    rows = len(indices)

    s = _Batch()
    s.case = case
    s.prefill = case["runs"] > 0
    s.groups = list(BLOCKS[case["block"]])
    if case["head"]:
        s.groups.append(ProjectionGroup("lm_head", ["lm_head"], s.groups[0].h_in, [case["head"]]))
    s.weights, s.x, s.y, s.calls = {}, {}, {}, []
    for g in s.groups:
        depth = 1 if g.name == "lm_head" else layers
        for name, h_out in zip(g.layer_names, g.sizes):
            s.weights[name] = _adapters(case, gen, g, h_out, depth)
        s.x[g.name] = _randn(gen, (rows, g.h_in), 1.0, dtype)
        s.y[g.name] = torch.zeros((depth, rows, g.h_out), dtype=dtype, device="cuda")
    for layer_id in range(layers):
        for g in s.groups:
            if g.name == "lm_head":
                continue
            base = _base(s.y[g.name][layer_id])
            if len(g.layer_names) > 1:
                linear = TensorParallelMultiAdapterLinear.load(base, layer_id, g.layer_names, g.sizes)
            else:
                linear = TensorParallelAdapterRowLinear.load(base, layer_id, g.layer_names[0])
            s.calls.append((linear, s.x[g.name]))
    if case["head"]:
        s.calls.append((MultiAdapterHead.load(_base(s.y["lm_head"][0]), 0, "lm_head"), s.x["lm_head"]))

    s.meta = make_meta(indices, torch.device("cuda", torch.cuda.current_device()))
    s.stacks, s.wrapper, s.graph = {}, None, None
    if case["kind"] == "stacked":
        s.stacks = stack_preloaded_adapters(s.weights, list(range(1, case["adapters"] + 1)))
        s.wrapper = PunicaWrapper(rows, rows, "cuda", True)
    if case["kind"] == "dropin":
        _plain_projections(s, rows)
    if case["graph"]:
        s.data = _tables(s)
        _forward(s)  # a server runs a step eagerly before it captures it
        torch.cuda.synchronize()
        s.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s.graph):
            _forward(s)
    for y in s.y.values():
        y.copy_(_randn(gen, y.shape, 1.0, dtype))
    return s


def _plain_projections(s, rows):
    """What a caller of the drop-in functions holds: one output per projection, and its own tables (built as here) over
    the reference's weight layouts."""
    s.data = _tables(s)
    s.y = {name: torch.zeros((s.case["layers"], rows, h_out), dtype=DTYPES[s.case["dtype"]], device="cuda")
           for g in s.groups for name, h_out in zip(g.layer_names, g.sizes)}
    s.input_of = {name: s.x[g.name] for g in s.groups for name in g.layer_names}
    for per_type in s.data.data.values():
        for rs in per_type[LORA].rank_data.values():
            rs.lora_a_ptr, rs.lora_b_ptr  # the tables, and the weights they point to, are laid out on first access


def _tables(s):
    if s.wrapper is not None:
        s.wrapper.update_metadata(s.meta, s.prefill)
    return AdapterBatchData.from_meta(s.meta, s.weights, s.stacks, s.wrapper, s.prefill)


def _forward(s):
    for linear, x in s.calls:
        linear(x, s.data)


def _forward_dropin(s):
    """LoraLinear's calls in the reference (utils/layers.py:107-167), projection by projection and rank by rank."""
    for layer_id in range(s.case["layers"]):
        for name, y in s.y.items():
            x = s.input_of[name]
            data = s.data.data.get(name)
            for r, rs in data[LORA].rank_data.items() if data is not None else ():
                if s.prefill:
                    v = sgmv.lora_a_sgmv_cutlass(x, rs.tmp_shrink, rs.lora_a_ptr, rs.segment_starts, rs.segment_ends,
                                                 layer_id, r)
                    sgmv.lora_b_sgmv_cutlass(y[layer_id], v, rs.tmp_expand, rs.lora_b_ptr, rs.segment_starts,
                                             rs.segment_ends, layer_id)
                else:
                    v = torch.zeros((x.size(0), r), dtype=x.dtype, device=x.device)
                    sgmv.add_lora_a_bgmv(v, x, rs.lora_a_ptr, rs.indices, layer_id)
                    sgmv.add_lora_b_bgmv(y[layer_id], v, rs.lora_b_ptr, rs.indices, layer_id)


def run(s):
    if s.graph is not None:
        s.graph.replay()
        return s.y
    if s.case["kind"] == "dropin":
        _forward_dropin(s)
        return s.y
    s.data = _tables(s)
    _forward(s)
    return s.y


def work(case):
    """Routed rows read x once per projection group and read and write y once; an adapter's A and B are read once per
    layer.  The intermediate of rank columns need not leave the chip."""
    e, rows, ranks = 2, _routed(case), _ranks(case)
    n = sum(rows.values())
    weighted = sum(rows[a] * ranks[a] for a in rows)
    touched = sum(ranks[a] for a in rows)
    moved = flops = 0
    groups = list(BLOCKS[case["block"]])
    if case["head"]:
        groups.append(ProjectionGroup("lm_head", ["lm_head"], groups[0].h_in, [case["head"]]))
    for g in groups:
        depth = 1 if g.name == "lm_head" else case["layers"]
        wide = len(g.sizes) * g.h_in + g.h_out
        moved += depth * e * (n * g.h_in + 2 * n * g.h_out + touched * wide)
        flops += depth * 2 * weighted * wide
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """Against the update in 64 bits without intermediate roundings, the outputs of these cases are off by 1.3e-3 to
    2.3e-3 of their norm in bf16 (largest single difference 1.2e-2) and by 2.0e-4 to 2.2e-4 in fp16 (9.3e-4): the
    roundings of the intermediate, of the update and of the sum.  Four times that."""
    return {"rel": 9e-3, "max": 5e-2} if case["dtype"] == "bf16" else {"rel": 9e-4, "max": 4e-3}
