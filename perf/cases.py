"""Workloads of the message-passing and attention paths, as programs of this framework run them.

Each case goes through ``tiga``'s public interface: a ``MessagePassing`` subclass called with a
graph and its fields, Torch autograd for the training steps, ``Graph.from_coo`` and
``Graph.transpose`` for graph construction.  Inputs are synthetic, made on the GPU from a seed.
"""

import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

# The package folder is not itself importable by name ("tiga-lang_amd").
sys.path.insert(1, os.path.join(os.getcwd(), "tiga-lang_amd"))

import tiga as tg  # noqa: E402

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
RMAT = (0.57, 0.19, 0.19, 0.05)
SLOPE = 0.2


# ---------------------------------------------------------------------------
# The user's kernels

class WeightedSum(tg.MessagePassing):
    reducer = tg.sum()

    def edge(self, src, dst, edge):
        return edge.weight * src.x


class GatAttention(tg.MessagePassing):
    reducer = tg.online_softmax()

    def edge(self, src, dst, edge, a_src, a_dst):
        score = F.leaky_relu((src.h * a_src).sum(-1) + (dst.h * a_dst).sum(-1), SLOPE)
        return self.reducer(score, src.h)


class DotAttention(tg.MessagePassing):
    reducer = tg.online_softmax()

    def edge(self, src, dst, edge, scale):
        return self.reducer((src.k * dst.q).sum(dim=-1) * scale, src.v)


class BiasedDotAttention(tg.MessagePassing):
    reducer = tg.online_softmax()

    def edge(self, src, dst, edge, scale):
        return self.reducer((src.k * dst.q).sum(dim=-1) * scale + edge.bias, src.v)


class ScoredAttention(tg.MessagePassing):
    reducer = tg.online_softmax()

    def __init__(self, net):
        super().__init__()
        self.net = tg.nn.trace(net)

    def edge(self, src, dst, edge):
        return self.reducer(self.net(edge.displacement, src.x, dst.x), src.x)


# ---------------------------------------------------------------------------
# What is measured

def listed():
    return [
        # A graph convolution's neighbour sum in training: 100,000 nodes of 16 neighbours,
        # hidden width 64, gradients of the features and of the edge weights.
        {"name": "sum-f32-w64-train", "op": "sum", "graph": "fixed", "nodes": 100_000,
         "degree": 16, "features": 64, "dtype": "f32", "train": True},
        # The same layer on raw input features of a width that fills no power of two, in
        # bfloat16, on a graph of uneven degrees.
        {"name": "sum-bf16-w100-train", "op": "sum", "graph": "poisson", "nodes": 200_000,
         "degree": 12, "features": 100, "dtype": "bf16", "train": True},
        # A wide first layer (bag-of-words features) of a mid-size graph.
        {"name": "sum-f32-w500-train", "op": "sum", "graph": "poisson", "nodes": 20_000,
         "degree": 8, "features": 500, "dtype": "f32", "train": True},
        # A classic attention layer (8 heads of 8) on a citation-size graph: all launches and
        # host time.
        {"name": "gat-f32-small-train", "op": "gat", "nodes": 2_700, "degree": 4, "heads": 8,
         "dim": 8, "dtype": "f32", "train": True},
        # The benchmark's headline: a million nodes, 17 million edges, 8 heads of 32.
        {"name": "gat-f32-1m-train", "op": "gat", "nodes": 1_000_000, "degree": 16, "heads": 8,
         "dim": 32, "dtype": "f32", "train": True},
        # Whole-graph inference of an attention layer in bfloat16 (no gradients kept).
        {"name": "gat-bf16-infer", "op": "gat", "nodes": 170_000, "degree": 14, "heads": 4,
         "dim": 64, "dtype": "bf16", "train": False},
        # Graph-transformer layer with an edge bias on a power-law graph (R-MAT scale 21).
        {"name": "dot-bf16-rmat21-train", "op": "dot", "graph": "rmat", "nodes": 1 << 21,
         "degree": 16, "heads": 4, "dim": 64, "dtype": "bf16", "bias": True, "train": True},
        # The same layer without a bias in inference, narrow heads, fp16, even degrees.
        {"name": "dot-f16-infer", "op": "dot", "graph": "poisson", "nodes": 300_000,
         "degree": 12, "heads": 8, "dim": 16, "dtype": "f16", "bias": False, "train": False},
        # Causal language-model attention over a packed batch of ragged sequences.
        {"name": "varlen-bf16-d128-train", "op": "attn", "kind": "varlen-causal",
         "sequences": 32, "min_len": 512, "max_len": 4096, "heads": 16, "dim": 128,
         "dtype": "bf16", "train": True},
        # Dense causal attention of one 4096-token sequence, lane-major fp16 tensors.
        {"name": "causal-f16-d64-infer", "op": "attn", "kind": "triangular", "sequences": 1,
         "min_len": 4096, "max_len": 4096, "heads": 16, "dim": 64, "dtype": "f16",
         "train": False},
        # Attention scored by a small network over [displacement | x_src | x_dst], training.
        {"name": "nn-f32-train", "op": "nn", "nodes": 131_072, "degree": 29.6, "width": 8,
         "hidden": 16, "train": True},
        # A power-law graph from an unordered edge list, and its transpose.
        {"name": "build-rmat20", "op": "build", "nodes": 1 << 20, "degree": 16,
         "index": "int64"},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choice(["sum", "sum", "gat", "gat", "dot", "dot", "attn", "attn", "nn", "build"])
    train = rng.random() < 0.6
    if op == "sum":
        nodes = _log_int(rng, 1_000, 500_000)
        degree = rng.randint(3, 32)
        width = _log_int(rng, 1, 600)
        width = max(1, min(width, int(1.5e9 / (nodes * degree))))
        graph = rng.choice(["fixed", "poisson", "rmat"])
        return {"op": "sum", "graph": graph, "nodes": _pow2(nodes) if graph == "rmat" else nodes,
                "degree": degree, "features": width, "dtype": rng.choice(["f32", "f32", "bf16",
                                                                          "f16"]),
                "train": train}
    if op == "gat":
        nodes = _log_int(rng, 1_000, 800_000)
        heads, dim = rng.choice([1, 2, 3, 4, 8]), rng.choice([8, 16, 32, 64, 128])
        degree = max(1, min(rng.randint(3, 24), int(3e9 / (nodes * heads * dim))))
        return {"op": "gat", "nodes": nodes, "degree": degree, "heads": heads, "dim": dim,
                "dtype": rng.choice(["f32", "f32", "bf16", "f16"]), "train": train}
    if op == "dot":
        nodes = _log_int(rng, 1_000, 800_000)
        heads, dim = rng.choice([1, 2, 4, 6, 8]), rng.choice([8, 16, 32, 64, 128])
        degree = max(1, min(rng.randint(3, 24), int(3e9 / (nodes * heads * dim))))
        graph = rng.choice(["poisson", "rmat"])
        return {"op": "dot", "graph": graph, "nodes": _pow2(nodes) if graph == "rmat" else nodes,
                "degree": degree, "heads": heads, "dim": dim,
                "dtype": rng.choice(["bf16", "f16", "f32"]), "bias": rng.random() < 0.5,
                "train": train}
    if op == "attn":
        kind = rng.choice(["varlen-causal", "varlen", "dense", "triangular"])
        heads, dim = rng.choice([1, 4, 8, 12, 16]), rng.choice([32, 64, 128])
        if kind in ("dense", "triangular"):
            n, low = 1, 0
            high = low = _log_int(rng, 100, 6_000)
        else:
            n, high = rng.randint(2, 48), _log_int(rng, 64, 4_096)
            n = max(2, min(n, int(3e8 / (high * high))))
            low = max(1, high // rng.choice([2, 8]))
        return {"op": "attn", "kind": kind, "sequences": n, "min_len": low, "max_len": high,
                "heads": heads, "dim": dim, "dtype": rng.choice(["bf16", "f16"]),
                "train": train}
    if op == "nn":
        return {"op": "nn", "nodes": _log_int(rng, 1_000, 150_000),
                "degree": round(rng.uniform(3.0, 30.0), 1), "width": rng.choice([4, 6, 8]),
                "hidden": rng.choice([8, 16, 20]), "train": True}
    return {"op": "build", "nodes": _pow2(_log_int(rng, 1_000, 1_500_000)),
            "degree": rng.randint(3, 16), "index": rng.choice(["int32", "int64"])}


def _pow2(n):
    return 1 << max(1, round(math.log2(n)))


# ---------------------------------------------------------------------------
# Inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _rmat_pairs(nodes, m, g):
    """(dst, src) of m R-MAT tuples, one quadrant draw per level."""
    scale = nodes.bit_length() - 1
    a, b, c, _ = RMAT
    dst = torch.zeros(m, dtype=torch.int64, device="cuda")
    src = torch.zeros(m, dtype=torch.int64, device="cuda")
    for level in range(scale):
        r = torch.rand(m, device="cuda", generator=g)
        dst |= (r >= a + b).to(torch.int64) << level
        src |= (((r >= a) & (r < a + b)) | (r >= a + b + c)).to(torch.int64) << level
    return dst, src


def _csr(case, g):
    """int64 (row_ptr, col) with sorted neighbour lists."""
    n, kind = case["nodes"], case.get("graph", "self-loop")
    if kind == "fixed":
        degree = case["degree"]
        col = torch.randint(0, n, (n, degree), device="cuda", generator=g).sort(dim=1)[0]
        return torch.arange(n + 1, dtype=torch.int64, device="cuda") * degree, col.reshape(-1)
    if kind == "rmat":
        # Duplicate edges are removed; more tuples than edges are drawn (small graphs repeat
        # more of theirs) and thinned evenly to nodes * degree.
        m = _edges(case)
        dst, src = _rmat_pairs(n, int(m * (1.15 if n >= 1 << 18 else 2 if n >= 1 << 13 else 5)),
                               g)
        keys = torch.unique(dst * n + src)
        pick = torch.arange(m, device="cuda") * keys.numel() // m
        keys = keys[pick]
    else:
        # Uniform pairs (in-degrees ~ Poisson), and for attention a self-loop per node.
        m = int(n * case["degree"])
        keys = torch.randint(0, n * n, (m,), device="cuda", generator=g)
        if kind == "self-loop":
            node = torch.arange(n, device="cuda")
            keys = torch.cat([keys, node * n + node])
        keys = keys.sort()[0]
    row_ptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    row_ptr[1:] = torch.cumsum(torch.bincount(keys // n, minlength=n), 0)
    return row_ptr, keys % n


def _lengths(case):
    """Sequence starts: the batch's shape, the same for every seed."""
    rng = np.random.default_rng([case["sequences"], case["max_len"]])
    lengths = rng.integers(case["min_len"], case["max_len"] + 1, size=case["sequences"])
    return np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)


def _inputs(case, seed):
    """The tensors of one case, as plain Torch."""
    g = _generator(seed)
    op = case["op"]
    randn = lambda *shape: torch.randn(*shape, device="cuda", generator=g)  # noqa: E731
    if op == "build":
        index = torch.int32 if case["index"] == "int32" else torch.int64
        dst, src = _rmat_pairs(case["nodes"], case["nodes"] * case["degree"], g)
        return {"dst": dst.to(index), "src": src.to(index)}
    if op == "attn":
        cu = _lengths(case)
        tokens, heads, dim = int(cu[-1]), case["heads"], case["dim"]
        dtype = DTYPES[case["dtype"]]
        if case["kind"] in ("dense", "triangular"):
            # [heads, tokens, dim] storage read as [tokens, heads, dim].
            make = lambda: randn(heads, tokens, dim).to(dtype).permute(1, 0, 2)  # noqa: E731
        else:
            make = lambda: randn(tokens, heads, dim).to(dtype)  # noqa: E731
        x = {"q": make(), "k": make(), "v": make(), "cu": cu}
        if case["train"]:
            x["dout"] = randn(tokens, heads, dim).to(dtype)
        return x
    row_ptr, col = _csr(case, g)
    x = {"row_ptr": row_ptr, "col": col}
    n, edges = case["nodes"], col.numel()
    if op == "nn":
        rows = torch.repeat_interleave(torch.arange(n, device="cuda"), row_ptr[1:] - row_ptr[:-1])
        pos = torch.rand(n, 3, device="cuda", generator=g)
        x["x"] = randn(n, case["width"])
        x["displacement"] = pos[col] - pos[rows]
        k, hidden = 3 + 2 * case["width"], case["hidden"]
        x["w1"], x["b1"] = randn(hidden, k) / math.sqrt(k), 0.1 * randn(hidden)
        x["w2"] = randn(1, hidden) / math.sqrt(hidden)
        x["dout"] = randn(n, case["width"])
        return x
    dtype = DTYPES[case["dtype"]]
    if op == "sum":
        x["x"] = randn(n, case["features"]).to(dtype)
        x["weight"] = torch.rand(edges, 1, device="cuda", generator=g).to(dtype)
        shape = (n, case["features"])
    else:
        shape = (n, case["heads"], case["dim"])
        if op == "gat":
            x["h"] = randn(*shape).to(dtype)
            x["a_src"] = 0.1 * randn(*shape[1:])
            x["a_dst"] = 0.1 * randn(*shape[1:])
        else:
            x["q"], x["k"], x["v"] = (randn(*shape).to(dtype) for _ in range(3))
            if case["bias"]:
                x["bias"] = randn(edges, case["heads"])
    if case["train"]:
        x["dout"] = randn(*shape).to(dtype)
    return x


_LEAVES = {"sum": ("x", "weight"), "gat": ("h", "a_src", "a_dst"), "dot": ("q", "k", "v", "bias"),
           "attn": ("q", "k", "v"), "nn": ("x", "displacement", "w1", "b1", "w2")}


def prepare(case, seed):
    x = _inputs(case, seed)
    op = case["op"]
    state = {"case": case}
    if op == "build":
        return {**state, **x}
    if op == "attn":
        n = int(x["cu"][-1])
        if case["kind"] == "dense":
            state["graph"] = tg.Graph.dense(n, device=torch.device("cuda"))
        elif case["kind"] == "triangular":
            state["graph"] = tg.Graph.triangular(n, device=torch.device("cuda"))
        else:
            state["graph"] = tg.Graph.cu_seqlens(torch.tensor(x["cu"], device="cuda"),
                                                 causal=case["kind"] == "varlen-causal")
        state["kernel"] = DotAttention()
    else:
        state["graph"] = tg.Graph.from_csr(x.pop("row_ptr"), x.pop("col"), num_src=case["nodes"])
    if op == "nn":
        # (No bias on the score: the softmax cancels it.)
        net = torch.nn.Sequential(torch.nn.Linear(3 + 2 * case["width"], case["hidden"]),
                                  torch.nn.LeakyReLU(SLOPE),
                                  torch.nn.Linear(case["hidden"], 1, bias=False)).cuda()
        with torch.no_grad():
            for p, name in zip(net.parameters(), ("w1", "b1", "w2")):
                p.copy_(x.pop(name))
        state["kernel"] = ScoredAttention(net)
        for p, name in zip(net.parameters(), ("w1", "b1", "w2")):
            x[name] = p
    elif op != "attn":
        state["kernel"] = {"sum": WeightedSum, "gat": GatAttention,
                           "dot": BiasedDotAttention if case.get("bias") else DotAttention}[op]()
    if case["train"]:
        leaves = [x[k] for k in _LEAVES[op] if k in x]
        for t in leaves:
            t.requires_grad_(True)
        state["leaves"] = leaves
    return {**state, **x}


# ---------------------------------------------------------------------------
# One pass

def _forward(s):
    case, kernel, graph = s["case"], s["kernel"], s["graph"]
    op = case["op"]
    if op == "sum":
        return kernel(graph=graph, src={"x": s["x"]}, dst={}, edge={"weight": s["weight"]})
    if op == "gat":
        return kernel(graph=graph, src={"h": s["h"]}, dst={"h": s["h"]}, a_src=s["a_src"],
                      a_dst=s["a_dst"])
    if op == "nn":
        return kernel(graph=graph, src={"x": s["x"]}, dst={"x": s["x"]},
                      edge={"displacement": s["displacement"]})
    edge = {"bias": s["bias"]} if "bias" in s else {}
    return kernel(graph=graph, src={"k": s["k"], "v": s["v"]}, dst={"q": s["q"]}, edge=edge,
                  scale=case["dim"] ** -0.5)


def run(state):
    case = state["case"]
    if case["op"] == "build":
        n = case["nodes"]
        graph = tg.Graph.from_coo(state["src"], state["dst"], num_src=n, num_dst=n)
        return [*graph.resolve_csr(), *graph.transpose().resolve_csr()]
    if not case["train"]:
        with torch.no_grad():
            return _forward(state)
    for t in state["leaves"]:
        t.grad = None
    out = _forward(state)
    out.backward(state["dout"])
    return [out.detach()] + [t.grad for t in state["leaves"]]


# ---------------------------------------------------------------------------
# What a pass cannot do without

def _edges(case):
    loops = 1 if case.get("graph", "self-loop") == "self-loop" else 0
    return int(case["nodes"] * (case["degree"] + loops))


def work(case):
    op = case["op"]
    if op == "build":
        size = 4 if case["index"] == "int32" else 8
        n, edges = case["nodes"], case["nodes"] * case["degree"]
        return {"bytes": size * (2 * edges + 2 * (n + 1 + edges)), "flops": 0}
    if op == "attn":
        lengths = np.diff(_lengths(case)).tolist()
        causal = case["kind"] in ("varlen-causal", "triangular")
        pairs = sum(n * (n + 1) / 2 if causal else n * n for n in lengths)
        width = case["heads"] * case["dim"]
        # Forward: two products; backward: S again, dP, dV, dK and dQ.
        tensors = 8 if case["train"] else 4
        return {"bytes": tensors * sum(lengths) * width * 2,
                "flops": (14 if case["train"] else 4) * pairs * width}
    n, edges = case["nodes"], _edges(case)
    index = 8 * (n + 1 + edges)
    if op == "nn":
        k, hidden, w = 3 + 2 * case["width"], case["hidden"], case["width"]
        return {"bytes": index + 4 * (2 * 3 * edges + 4 * n * w),
                "flops": edges * (6 * (k * hidden + hidden) + 6 * w)}
    size = torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
    if op == "sum":
        width = case["features"]
        if case["train"]:
            return {"bytes": index + size * (2 * edges + 4 * n * width),
                    "flops": 6 * edges * width}
        return {"bytes": index + size * (edges + 2 * n * width), "flops": 2 * edges * width}
    width = case["heads"] * case["dim"]
    if op == "gat":
        return {"bytes": index + size * n * width * (4 if case["train"] else 2),
                "flops": edges * width * (8 if case["train"] else 2)}
    bias = 4 * edges * case["heads"] if case["bias"] else 0
    return {"bytes": index + bias * (2 if case["train"] else 1) +
            size * n * width * (8 if case["train"] else 4),
            "flops": edges * width * (14 if case["train"] else 4)}


def tolerance(case):
    if case["op"] == "build":
        return "exact"
    dtype = case.get("dtype", "f32")
    if dtype != "f32":
        return {"rel": 1e-2 if dtype == "bf16" else 1.5e-3}
    # A score's sign at the leaky ReLU's kink is a matter of rounding, and its gradient jumps
    # there: about 1e-4 of the gradients' norm on a million nodes.
    return {"rel": 5e-4 if case["op"] in ("gat", "nn") else 2e-6}


# ---------------------------------------------------------------------------
# The same in 64 bits

def _segment_softmax(score, row, n):
    """Softmax weights of [edges, heads] scores over each of n rows."""
    top = torch.full((n, score.shape[1]), -math.inf, dtype=score.dtype, device=score.device)
    top = top.scatter_reduce(0, row[:, None].expand_as(score), score.detach(), "amax")
    p = torch.exp(score - top[row])
    total = torch.zeros_like(top).index_add(0, row, p)
    return p / total[row]


def _row_chunks(row_ptr, most):
    """Ranges of rows with about `most` edges each."""
    ends = row_ptr.cpu().numpy()
    r, n = 0, len(ends) - 1
    while r < n:
        stop = int(np.searchsorted(ends, ends[r] + most, side="right")) - 1
        stop = min(max(stop, r + 1), n)
        yield r, stop, int(ends[r]), int(ends[stop])
        r = stop


def _exact_csr(case, x):
    """Rows in chunks: forward and, by autograd, the gradients of each chunk."""
    op, n, train = case["op"], case["nodes"], case["train"]
    row_ptr, col = x["row_ptr"], x["col"]
    # Read whole by every chunk; the others (per edge, or per destination) are cut.
    whole = {"sum": ("x",), "gat": ("h", "a_src", "a_dst"), "dot": ("k", "v"),
             "nn": ("x", "w1", "b1", "w2")}[op]
    per_edge = {"sum": "weight", "dot": "bias", "nn": "displacement"}.get(op)
    full = {k: x[k].double().requires_grad_(train) for k in whole}
    grads = {k: torch.zeros_like(v) for k, v in full.items()}
    width = math.prod(next(iter(full.values())).shape[1:]) if op != "nn" else 32
    outs, cut = [], {}
    for r0, r1, e0, e1 in _row_chunks(row_ptr, max(1, int(2.5e8 / width))):
        rows = r1 - r0
        row = torch.repeat_interleave(torch.arange(rows, device="cuda"),
                                      row_ptr[r0 + 1:r1 + 1] - row_ptr[r0:r1])
        j = col[e0:e1]
        part = {}
        if per_edge in x:
            part[per_edge] = x[per_edge][e0:e1].double().requires_grad_(train)
        if op == "dot":
            part["q"] = x["q"][r0:r1].double().requires_grad_(train)
        if op == "sum":
            message = part["weight"] * full["x"][j]
        elif op == "gat":
            hj = full["h"][j]
            score = F.leaky_relu((hj * full["a_src"]).sum(-1) +
                                 (full["h"][r0:r1] * full["a_dst"]).sum(-1)[row], SLOPE)
            message = _segment_softmax(score, row, rows)[..., None] * hj
        elif op == "dot":
            score = (full["k"][j] * part["q"][row]).sum(-1) * case["dim"] ** -0.5
            if case["bias"]:
                score = score + part["bias"]
            message = _segment_softmax(score, row, rows)[..., None] * full["v"][j]
        else:
            fields = torch.cat([part["displacement"], full["x"][j], full["x"][r0:r1][row]], 1)
            hidden = F.leaky_relu(fields @ full["w1"].t() + full["b1"], SLOPE)
            score = hidden @ full["w2"].t()
            message = _segment_softmax(score, row, rows) * full["x"][j]
        out = torch.zeros((rows, *message.shape[1:]), dtype=torch.float64,
                          device="cuda").index_add(0, row, message)
        outs.append(out.detach())
        if train:
            names = list(full) + list(part)
            got = torch.autograd.grad(out, [*full.values(), *part.values()],
                                      x["dout"][r0:r1].double())
            for k, v in zip(names, got):
                if k in full:
                    grads[k] += v
                else:
                    cut.setdefault(k, []).append(v)
    out = torch.cat(outs)
    if not train:
        return out
    grads.update({k: torch.cat(v) for k, v in cut.items()})
    return [out] + [grads[k] for k in _LEAVES[op] if k in grads]


def _exact_attn(case, x):
    causal = case["kind"] in ("varlen-causal", "triangular")
    scale = case["dim"] ** -0.5
    cu = x["cu"]
    names = ("out", "q", "k", "v") if case["train"] else ("out",)
    got = {k: torch.empty(int(cu[-1]), case["heads"], case["dim"], dtype=torch.float64,
                          device="cuda") for k in names}
    for s, e in zip(cu[:-1].tolist(), cu[1:].tolist()):
        if e == s:
            continue
        lanes = lambda t: t[s:e].double().permute(1, 0, 2).contiguous()  # noqa: E731
        q, k, v = lanes(x["q"]), lanes(x["k"]), lanes(x["v"])
        p = (q @ k.transpose(1, 2)) * scale
        if causal:
            p.masked_fill_(torch.ones(e - s, e - s, dtype=torch.bool, device="cuda").triu(1),
                           -math.inf)
        p = torch.softmax(p, -1)
        got["out"][s:e] = (p @ v).permute(1, 0, 2)
        if not case["train"]:
            continue
        dout = lanes(x["dout"])
        got["v"][s:e] = (p.transpose(1, 2) @ dout).permute(1, 0, 2)
        dp = dout @ v.transpose(1, 2)
        dp = p * (dp - (p * dp).sum(-1, keepdim=True)) * scale
        got["q"][s:e] = (dp @ k).permute(1, 0, 2)
        got["k"][s:e] = (dp.transpose(1, 2) @ q).permute(1, 0, 2)
    return [got[k] for k in names] if case["train"] else got["out"]


def exact(case, seed):
    if case["op"] == "build":
        return None
    x = _inputs(case, seed)
    with torch.enable_grad():
        return _exact_attn(case, x) if case["op"] == "attn" else _exact_csr(case, x)
