"""The encoder's work as its users have it: the cases whose time is looked at, and how to make and run one.

A case is one padding-free BERT encoder over one batch that is on the GPU already:

  entry    the public way in: "encoder" (EffectiveTransformerEncoder, the weights kept by the object), "ids" (the same object
           from token ids, embedding block included), "graph" (the encoder captured once, replayed on each batch's tensors) or
           "ops" (the registered Input / Layer / Output ops, weights handed to every call as the reference's op takes them)
  dtype    "fp16" or "fp32", both types of the op
  layers, heads   the model: heads * 64 hidden, 4 * hidden in the feed-forward part (sample/bert_config.json: 12 and 12)
  batch, seq      the padded batch
  lo, hi          the sequences' lengths, evenly spread over lo .. hi
  long_share      0, or that share of the sequences is lengthened to 3/4 seq .. seq (skewed batches)
"""
import math

import torch

import effective_transformer_amd as et
from effective_transformer_amd import ops, torch_ops

HEAD = 64
VOCAB, TYPES = 30522, 2


def _case(name, entry, dtype, layers, heads, batch, seq, lo, hi, long_share=0.0):
    return {"name": name, "entry": entry, "dtype": dtype, "layers": layers, "heads": heads, "batch": batch, "seq": seq,
            "lo": lo, "hi": hi, "long_share": long_share}


def listed():
    return [
        # one user's query, answered at once: latency, launches and host work
        _case("one_query", "encoder", "fp16", 12, 12, 1, 32, 8, 32),
        # a handful of requests of mixed length that arrived together, from token ids
        _case("few_requests_ids", "ids", "fp16", 12, 12, 8, 128, 16, 128),
        # one fp32 layer on a small batch: the first configuration of the benchmark, the unit a caller tests with
        _case("one_layer_fp32", "encoder", "fp32", 1, 12, 8, 32, 8, 32),
        # a serving loop that replays a captured graph on each batch it collects
        _case("serving_graph", "graph", "fp16", 12, 12, 16, 64, 16, 64),
        # the small end of the published fp16 table
        _case("base_100x32", "encoder", "fp16", 12, 12, 100, 32, 8, 32),
        # the op-level drop-in inside somebody else's graph, odd batch and odd padded length
        _case("ops_217x53", "ops", "fp16", 12, 12, 217, 53, 13, 53),
        # the headline batch
        _case("base_1000x64", "encoder", "fp16", 12, 12, 1000, 64, 16, 64),
        # the large end of the published fp32 table
        _case("fp32_500x64", "encoder", "fp32", 12, 12, 500, 64, 16, 64),
        # the large model on a batch of very unequal lengths
        _case("large_skewed_256x128", "encoder", "fp16", 24, 16, 256, 128, 8, 32, 0.3),
        # documents
        _case("documents_32x512", "encoder", "fp16", 12, 12, 32, 512, 256, 512),
        # the longest sequences the op takes
        _case("longest_16x1024", "encoder", "fp16", 12, 12, 16, 1024, 376, 1024),
        # fp32 passages of odd padded length, odd batch
        _case("fp32_passages_15x379", "encoder", "fp32", 12, 12, 15, 379, 131, 379),
    ]


def _lengths(case, generator):
    """One length from each of `batch` equal slices of lo .. hi, in random order, so that another seed has other lengths and
    nearly the same total; host tensor."""
    n, lo, hi = case["batch"], case["lo"], case["hi"]
    u = (torch.arange(n) + torch.rand(n, generator=generator)) / n
    lens = lo + (u * (hi - lo + 1)).long().clamp(max=hi - lo)
    lens = lens[torch.randperm(n, generator=generator)]
    m = round(case["long_share"] * n)
    if m:
        low = 3 * case["seq"] // 4
        lens[torch.randperm(n, generator=generator)[:m]] = low + (torch.rand(m, generator=generator) * (case["seq"] - low + 1)).long().clamp(max=case["seq"] - low)
    return lens


def _tokens(case):
    """Expected (sum of the lengths, sum of their squares)."""
    def moments(lo, hi):
        n = hi - lo + 1
        return (lo + hi) / 2.0, sum(v * v for v in range(lo, hi + 1)) / n
    m1, m2 = moments(case["lo"], case["hi"])
    l1, l2 = moments(3 * case["seq"] // 4, case["seq"])
    s = case["long_share"]
    return case["batch"] * ((1 - s) * m1 + s * l1), case["batch"] * ((1 - s) * m2 + s * l2)


def work(case):
    """Bytes: the valid rows of the input (ids: the table rows and the ids), the masks of the valid queries, the weights and the
    padded output, once each.  Operations: the products of the valid rows with the weights, and of each sequence with itself."""
    e = 2 if case["dtype"] == "fp16" else 4
    hidden, layers, positions = case["heads"] * HEAD, case["layers"], case["batch"] * case["seq"]
    tokens, squares = _tokens(case)
    nbytes = tokens * hidden * e + 4 * positions + tokens * case["seq"] * e + layers * (12 * hidden * hidden + 13 * hidden) * e
    nbytes += positions * hidden * e
    if case["entry"] == "ids":
        nbytes += 8 * tokens + (TYPES + case["seq"] + 2) * hidden * e
    return {"bytes": nbytes, "flops": layers * (24.0 * tokens * hidden * hidden + 4.0 * squares * hidden)}


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    case = _case("", rng.choice(("encoder", "encoder", "encoder", "ids", "graph", "ops")),
                 rng.choice(("fp16", "fp16", "fp16", "fp32")), rng.choice((1, 6, 12, 12, 12, 24)), rng.choice((8, 12, 12, 16)), 1,
                 spread(16, 1024), 1, 1)
    del case["name"]
    if case["entry"] == "ids":
        case["seq"] = min(case["seq"], 512)
    case["batch"] = max(1, min(1000, spread(32, 64000) // case["seq"]))
    case["hi"] = case["seq"]
    case["lo"] = max(1, int(case["seq"] * rng.uniform(0.1, 0.9)))
    if rng.random() < 0.2:
        case["lo"], case["hi"], case["long_share"] = max(1, case["seq"] // 16), max(1, case["seq"] // 4), 0.3
    most = max(work(c)["flops"] for c in listed() if c["dtype"] == case["dtype"])
    while work(case)["flops"] > most:
        case["batch"] = max(1, case["batch"] * 3 // 4)
        if case["batch"] == 1:
            case["layers"] = 1
    return case


def _layer_weights(case, dtype, generator):
    """The 16 tensors of each layer in the order of the reference's weights_value (kernels N(0, 0.02))."""
    hidden = case["heads"] * HEAD

    def kernel(k, n):
        return torch.randn(k, n, device="cuda", dtype=dtype, generator=generator).mul_(0.02)

    def vector(n, base, width):
        return torch.randn(n, device="cuda", dtype=dtype, generator=generator).mul_(width).add_(base)

    layers = []
    for _ in range(case["layers"]):
        w = []
        for _ in range(4):
            w += [kernel(hidden, hidden), vector(hidden, 0.0, 0.02)]
        w += [vector(hidden, 0.0, 0.05), vector(hidden, 1.0, 0.05)]
        w += [kernel(hidden, 4 * hidden), vector(4 * hidden, 0.0, 0.02), kernel(4 * hidden, hidden), vector(hidden, 0.0, 0.02)]
        w += [vector(hidden, 0.0, 0.05), vector(hidden, 1.0, 0.05)]
        layers.append(w)
    return layers


def prepare(case, seed):
    dtype = torch.float16 if case["dtype"] == "fp16" else torch.float32
    batch, seq, heads = case["batch"], case["seq"], case["heads"]
    hidden = heads * HEAD
    host = torch.Generator().manual_seed(int(seed))
    gpu = torch.Generator(device="cuda").manual_seed(int(seed))
    lens = _lengths(case, host).cuda()
    mask = (torch.arange(seq, device="cuda")[None, :] < lens[:, None]).to(torch.int32).contiguous()
    attention = mask[:, None, :].expand(batch, seq, seq).to(dtype).contiguous()
    state = {"case": case, "mask": mask, "attention": attention}
    layers = _layer_weights(case, dtype, gpu)
    if case["entry"] == "ops":
        state["weights"] = layers
    else:
        flat = [t for w in layers for t in w]
        state["encoder"] = et.EffectiveTransformerEncoder(case["layers"], heads, HEAD, flat, dtype)
    if case["entry"] == "ids":
        def table(n):
            return torch.randn(n, hidden, device="cuda", dtype=dtype, generator=gpu).mul_(0.02)
        state["embeddings"] = ops.EmbeddingWeights(
            torch.device("cuda"), dtype, table(VOCAB), table(1)[0].add_(1.0), table(1)[0], token_type_embeddings=table(TYPES),
            position_embeddings=table(512))
        state["ids"] = torch.randint(0, VOCAB, (batch, seq), device="cuda", dtype=torch.int32, generator=gpu)
        state["types"] = torch.randint(0, TYPES, (batch, seq), device="cuda", dtype=torch.int32, generator=gpu)
    else:
        state["x"] = torch.randn(batch, seq, hidden, device="cuda", dtype=dtype, generator=gpu)
    if case["entry"] == "graph":
        state["graph"] = state["encoder"].make_graph(state["x"], mask, attention)
    return state


def run(state):
    entry = state["case"]["entry"]
    if entry == "ids":
        return state["encoder"].forward_ids(state["ids"], state["types"], state["mask"], state["attention"], state["embeddings"])
    if entry == "graph":
        return state["graph"](state["x"], state["mask"], state["attention"])
    if entry == "ops":
        return torch_ops.encoder(state["x"], state["mask"], state["attention"], state["weights"], state["case"]["heads"], HEAD)
    return state["encoder"](state["x"], state["mask"], state["attention"])


def tolerance(case):
    """fp16: each of a layer's seven results is rounded to 11 bits and the errors add up over the layers; the largest of some
    millions of values is off by about ten times the mean.  fp32: 24-bit values and sums."""
    if case["dtype"] == "fp16":
        return {"rel": 5e-3, "max": 5e-2}
    return {"rel": 1e-5, "max": 2e-4}
