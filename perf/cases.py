"""Performance cases: what a program that uses fastmoe_amd has it do, over the range it does it in.

Five kinds of call, each through the package's public entry points:

  combine   ``grouped_weighted_scatter_add`` over a list of ragged expert buffers, or
            ``weighted_scatter_add`` over one packed buffer (E = 1 list, ``packed``); forward only
            under ``no_grad`` (inference) or forward + backward with every gradient (training)
  inplace   ``out.zero_()`` and the accumulating call with prepared metadata, captured in a HIP
            graph and replayed: the way the kernel benchmark of the operator runs it
  dispatch  ``permute_tokens``: routing slots grouped by expert and the token rows gathered, forward
            only or with its backward
  layer     ``MoEFeedForward``: router, permutation, expert MLPs and combine, forward + backward
  reduce    ``weighted_scatter_add(mode="atomic")``: many rows into few output rows, the use that
            the atomic mode is documented for

Routing follows the layer's own producer: random router logits (for ``zipf`` with a per-expert bias,
so that a few experts take most rows), top-k, fp32 softmax over the chosen, slots sorted by expert.
"""
import math

import torch

import fastmoe_amd
from fastmoe_amd.workloads import zipf_bias

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16,
          "int64": torch.int64, "int32": torch.int32}
BYTES = {"fp32": 4, "bf16": 2, "fp16": 2, "int64": 8, "int32": 4}

# The largest listed case moves this many bytes; a drawn one at most as many.
MOST_BYTES = 3.5e9


def _combine(name, T, D, E, k, dtype, gates, index="int64", routing="topk", grad=False,
             packed=False):
    return {"name": name, "kind": "combine", "T": T, "D": D, "E": E, "k": k, "dtype": dtype,
            "gates": gates, "index": index, "routing": routing, "grad": grad, "packed": packed}


def listed():
    return [
        # One decoding step of a few sequences: the smallest calls, all latency and launches.
        _combine("decode", 8, 7168, 256, 8, "bf16", "bf16"),
        # A small fp32 training step (the plumbing configuration).
        _combine("small-step", 256, 512, 8, 2, "fp32", "fp32", grad=True),
        # Prefill, forward only: the mid configuration.
        _combine("prefill", 8192, 4096, 64, 6, "bf16", "fp32"),
        # Prefill with a skewed router: a few experts hold most of the rows.
        _combine("prefill-skewed", 16384, 7168, 256, 8, "bf16", "bf16", routing="zipf"),
        # A training micro-batch on one rank of an expert-parallel group: 32 local experts.
        _combine("rank-step", 1024, 7168, 32, 8, "bf16", "fp32", grad=True),
        # The headline training step: D = 16384, 256 experts, top-8, one packed buffer.
        _combine("packed-step", 4096, 16384, 256, 8, "bf16", "fp32", grad=True, packed=True),
        # Odd everything: token count, hidden size, experts; fp16 and int32 indices.
        _combine("odd-step", 3001, 1001, 13, 3, "fp16", "fp16", "int32", grad=True),
        # The operator's own kernel benchmark: fp32, 256 experts of 64 rows, uniform indices.
        {"name": "inplace-graph", "kind": "inplace", "T": 4096, "D": 16384, "E": 256, "k": 4,
         "dtype": "fp32"},
        # Dispatch of one decoding step.
        {"name": "dispatch-decode", "kind": "dispatch", "T": 32, "D": 7168, "E": 256, "k": 8,
         "dtype": "bf16", "gates": "bf16", "grad": False},
        # Dispatch in training, forward and backward.
        {"name": "dispatch-step", "kind": "dispatch", "T": 8192, "D": 4096, "E": 64, "k": 6,
         "dtype": "bf16", "gates": "fp32", "grad": True},
        # The whole layer, forward and backward (its expert MLPs are library products).
        {"name": "layer-step", "kind": "layer", "T": 2048, "D": 2048, "F": 1024, "E": 16, "k": 2,
         "dtype": "bf16"},
        # Reduction-like scatter into few rows.
        {"name": "reduce", "kind": "reduce", "T": 128, "D": 1024, "N": 65536, "dtype": "fp32"},
    ]


def _log(rng, lo, hi):
    """An integer between lo and hi, spread evenly over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _hidden(rng, lo=512, hi=16384, odd=0.25):
    """A hidden size: usually a multiple of 64, sometimes of 8, sometimes any number."""
    d = _log(rng, lo, hi)
    if rng.random() < odd:
        return d
    return max(64, d // 64 * 64) if rng.random() < 0.8 else d // 8 * 8


def draw(rng):
    while True:
        kind = rng.choice(["combine"] * 6 + ["dispatch"] * 3 + ["inplace", "layer", "reduce"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        if kind == "combine":
            grad = rng.random() < 0.5
            packed = grad and rng.random() < 0.3
            E = _log(rng, 2, 256 if packed or not grad else 56)
            c = _combine("", _log(rng, 1, 16384), _hidden(rng), E, rng.randint(1, min(8, E)),
                         dtype, rng.choice([dtype, "fp32"]), rng.choice(["int64", "int64", "int32"]),
                         rng.choice(["topk", "topk", "zipf"]), grad, packed)
        elif kind == "inplace":
            c = {"kind": kind, "T": _log(rng, 256, 8192), "D": _hidden(rng, odd=0.1),
                 "E": _log(rng, 8, 256), "k": rng.randint(1, 8),
                 "dtype": rng.choice(["fp32", "fp32", "bf16"])}
        elif kind == "dispatch":
            E = _log(rng, 2, 256)
            c = {"kind": kind, "T": _log(rng, 1, 16384), "D": _hidden(rng), "E": E,
                 "k": rng.randint(1, min(8, E)), "dtype": dtype,
                 "gates": rng.choice([dtype, "fp32"]), "grad": rng.random() < 0.5}
        elif kind == "layer":
            c = {"kind": kind, "T": _log(rng, 256, 4096), "D": _hidden(rng, 256, 2048, 0.0),
                 "F": _hidden(rng, 256, 2048, 0.0), "E": rng.choice([4, 8, 16]),
                 "k": rng.randint(1, 4), "dtype": "bf16"}
        else:
            c = {"kind": kind, "T": _log(rng, 16, 1024), "D": _hidden(rng, 64, 2048),
                 "N": _log(rng, 4096, 131072), "dtype": rng.choice(["fp32", "fp32", "bf16"])}
        c.pop("name", None)
        if work(c)["bytes"] <= MOST_BYTES:
            return c


# ---- inputs ---------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(shape, dtype, gen):
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


def _topk(case, gen):
    """(expert ids int64 [T, k], fp32 gates [T, k]): the top-k of random router logits (one draw per
    case, so that an expert has the same number of rows for every seed), its tokens shuffled and
    their gates drawn anew."""
    base = _gen(1)
    logits = torch.randn(case["T"], case["E"], generator=base, device="cuda")
    if case.get("routing") == "zipf":
        logits += torch.from_numpy(zipf_bias(case["E"], 1)).cuda()
    ids = torch.topk(logits, case["k"], dim=-1).indices
    ids = ids[torch.randperm(case["T"], generator=gen, device="cuda")]
    gates = torch.softmax(torch.randn(ids.shape, generator=gen, device="cuda"), dim=-1)
    return ids, gates


def _combine_inputs(case, seed):
    """Packed rows [N, D], scatter index, gates, rows per expert and the output's gradient."""
    gen = _gen(seed)
    ids, gates = _topk(case, gen)
    flat = ids.reshape(-1)
    order = torch.argsort(flat, stable=True)
    idx = (order // case["k"]).to(DTYPES[case["index"]])
    w = gates.reshape(-1)[order].to(DTYPES[case["gates"]])
    counts = torch.bincount(flat, minlength=case["E"]).tolist()
    dtype = DTYPES[case["dtype"]]
    x = _normal((idx.numel(), case["D"]), dtype, gen)
    go = _normal((case["T"], case["D"]), dtype, gen) if case["grad"] else None
    return x, idx, w, counts, go


def _inplace_inputs(case, seed):
    """As the kernel benchmark: equal experts, uniform indices and gates."""
    gen = _gen(seed)
    rows = max(1, case["T"] * case["k"] // case["E"])
    n = rows * case["E"]
    idx = torch.randint(0, case["T"], (n,), generator=gen, device="cuda")
    w = torch.rand(n, generator=gen, device="cuda")
    x = _normal((n, case["D"]), DTYPES[case["dtype"]], gen)
    return x, idx, w, [rows] * case["E"]


def _dispatch_inputs(case, seed):
    gen = _gen(seed)
    ids, gates = _topk(case, gen)
    gates = gates.to(DTYPES[case["gates"]])
    dtype = DTYPES[case["dtype"]]
    x = _normal((case["T"], case["D"]), dtype, gen)
    if not case["grad"]:
        return x, ids, gates, None, None
    n = case["T"] * case["k"]
    return (x, ids, gates, _normal((n, case["D"]), dtype, gen),
            _normal((n,), DTYPES[case["gates"]], gen))


def _layer_inputs(case, seed):
    """Layer input, output gradient and the weights in parameter order."""
    gen = _gen(seed)
    dtype = DTYPES[case["dtype"]]
    D, F, E = case["D"], case["F"], case["E"]
    x = _normal((1, case["T"], D), dtype, gen)
    go = _normal((1, case["T"], D), dtype, gen)
    weights = [_normal((E, D), torch.float32, gen).mul_(D ** -0.5).to(dtype)]
    for _ in range(E):
        weights.append(_normal((F, D), torch.float32, gen).mul_(D ** -0.5).to(dtype))
        weights.append(_normal((D, F), torch.float32, gen).mul_(F ** -0.5).to(dtype))
    return x, go, weights


def _reduce_inputs(case, seed):
    gen = _gen(seed)
    idx = torch.randint(0, case["T"], (case["N"],), generator=gen, device="cuda")
    w = torch.rand(case["N"], generator=gen, device="cuda")
    return _normal((case["N"], case["D"]), DTYPES[case["dtype"]], gen), idx, w


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind == "combine":
        x, idx, w, counts, s["go"] = _combine_inputs(case, seed)
        grad = case["grad"]
        # the experts' outputs are separate allocations, as separate modules return them
        xs = [x] if case["packed"] else [c.clone() for c in x.split(counts)]
        s["xs"] = [t.requires_grad_(grad) for t in xs]
        s["idx"], s["w"] = idx, w.requires_grad_(grad)
    elif kind == "inplace":
        x, idx, w, counts = _inplace_inputs(case, seed)
        xs = [c.clone() for c in x.split(counts)]
        out = torch.zeros(case["T"], case["D"], dtype=x.dtype, device="cuda")
        meta = fastmoe_amd.prepare_grouped_metadata(xs, "cuda")

        def step():
            out.zero_()
            fastmoe_amd.grouped_weighted_scatter_add(xs, idx, w, out.shape, out=out, metadata=meta)

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            step()
        s.update(graph=graph, out=out, keep=(xs, idx, w, meta))
    elif kind == "dispatch":
        x, ids, gates, g_rows, g_gates = _dispatch_inputs(case, seed)
        s.update(x=x.requires_grad_(case["grad"]), ids=ids,
                 gates=gates.requires_grad_(case["grad"]), g_rows=g_rows, g_gates=g_gates)
    elif kind == "layer":
        x, go, weights = _layer_inputs(case, seed)
        with torch.device("cuda"):
            layer = fastmoe_amd.MoEFeedForward(case["D"], case["F"], case["E"], case["k"])
        layer = layer.to(x.dtype)
        with torch.no_grad():
            for p, v in zip(layer.parameters(), weights):
                p.copy_(v)
        s.update(layer=layer, params=list(layer.parameters()), x=x.requires_grad_(True), go=go)
    else:
        s["x"], s["idx"], s["w"] = _reduce_inputs(case, seed)
    return s


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "combine":
        shape = (case["T"], case["D"])
        if not case["grad"]:
            with torch.no_grad():
                return fastmoe_amd.grouped_weighted_scatter_add(s["xs"], s["idx"], s["w"], shape)
        if case["packed"]:
            out = fastmoe_amd.weighted_scatter_add(s["xs"][0], s["idx"], s["w"], shape)
        else:
            out = fastmoe_amd.grouped_weighted_scatter_add(s["xs"], s["idx"], s["w"], shape)
        return [out.detach(), *torch.autograd.grad(out, [s["w"], *s["xs"]], s["go"])]
    if kind == "inplace":
        s["graph"].replay()
        return s["out"]
    if kind == "dispatch":
        p = fastmoe_amd.permute_tokens(s["x"], s["ids"], s["gates"], case["E"])
        outs = [p.permuted_data.detach(), p.expert_counts, p.reverse_map_indices,
                p.sorted_weights.detach(), p.expert_offsets, p.slot_pos]
        if not case["grad"]:
            return outs
        return outs + list(torch.autograd.grad([p.permuted_data, p.sorted_weights],
                                               [s["x"], s["gates"]], [s["g_rows"], s["g_gates"]]))
    if kind == "layer":
        out = s["layer"](s["x"])
        return [out.detach(), *torch.autograd.grad(out, [s["x"], *s["params"]], s["go"],
                                                   allow_unused=True)]
    with torch.no_grad():
        return fastmoe_amd.weighted_scatter_add(s["x"], s["idx"], s["w"], (case["T"], case["D"]),
                                                mode="atomic")


def work(case):
    """Bytes and operations of one pass.  Forward and backward are two calls with the rest of a
    model between them, so each reads its own inputs once and writes its own outputs once."""
    kind, T, D, b = case["kind"], case["T"], case["D"], BYTES[case["dtype"]]
    if kind == "combine":
        n = T * case["k"]
        routing = n * (BYTES[case["index"]] + BYTES[case["gates"]])
        nbytes, flops = n * D * b + T * D * b + routing, 2 * n * D
        if case["grad"]:
            nbytes += T * D * b + 2 * n * D * b + routing + n * BYTES[case["gates"]]
            flops += 3 * n * D
    elif kind == "inplace":
        n = max(1, T * case["k"] // case["E"]) * case["E"]
        nbytes, flops = n * D * b + T * D * b + n * 12, 2 * n * D
    elif kind == "dispatch":
        n, g = T * case["k"], BYTES[case["gates"]]
        nbytes, flops = T * D * b + n * D * b + n * (8 + 2 * g + 8 + 4), 0
        if case["grad"]:
            nbytes += n * D * b + T * D * b + n * (4 + 2 * g)
            flops += n * D
    elif kind == "layer":
        n, F, E = T * case["k"], case["F"], case["E"]
        weights = E * D + 2 * E * D * F
        nbytes = (3 * weights + 4 * T * D) * b  # weights twice, their gradients; x, out and theirs
        flops = 3 * (4 * n * D * F + 2 * T * D * E) + 8 * n * D
    else:
        nbytes, flops = case["N"] * D * b + T * D * b + case["N"] * 12, 2 * case["N"] * D
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    """About four times what the types' own rounding shows: a result summed in fp32 and rounded
    once (bf16: half of 2^-8 of a value at most, 1.7e-3 in the 2-norm; fp16: an eighth of that;
    fp32: sums of a few terms).  A dispatch without its backward moves bits and
    counts.  The layer rounds to bf16 after every product."""
    if case["kind"] == "dispatch" and not case["grad"]:
        return "exact"
    if case["kind"] == "layer":
        return {"rel": 2e-2}
    if case["dtype"] == "bf16":
        return {"rel": 7e-3, "max": 1.6e-2}
    if case["dtype"] == "fp16":
        return {"rel": 9e-4, "max": 2e-3}
    if case["kind"] == "reduce":  # hundreds to thousands of terms, in any order
        return {"rel": 2e-6, "max": 1e-5}
    return {"rel": 4e-7, "max": 4e-6}


# ---- the same in 64 bits ------------------------------------------------------------------------


def _sum_rows(x, idx, w, T):
    """out[idx[g]] += w[g] * x[g] in fp64, in column blocks."""
    out = torch.zeros(T, x.shape[1], dtype=torch.float64, device=x.device)
    idx, w = idx.long(), w.double()[:, None]
    for c in range(0, x.shape[1], 2048):
        out[:, c:c + 2048] = torch.zeros_like(out[:, c:c + 2048]).index_add_(
            0, idx, x[:, c:c + 2048].double() * w)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "combine":
        x, idx, w, counts, go = _combine_inputs(case, seed)
        out = _sum_rows(x, idx, w, case["T"])
        if not case["grad"]:
            return out
        i = idx.long()
        gx = go.double()[i] * w.double()[:, None]
        gw = torch.zeros(i.numel(), dtype=torch.float64, device=x.device)
        for c in range(0, x.shape[1], 2048):
            gw += (go[:, c:c + 2048].double()[i] * x[:, c:c + 2048].double()).sum(1)
        return [out, gw, *([gx] if case["packed"] else gx.split(counts))]
    if kind == "inplace":
        x, idx, w, _ = _inplace_inputs(case, seed)
        return _sum_rows(x, idx, w, case["T"])
    if kind == "dispatch":
        x, ids, gates, g_rows, g_gates = _dispatch_inputs(case, seed)
        if not case["grad"]:
            return None
        order = torch.argsort(ids.reshape(-1), stable=True)
        rev = order // case["k"]
        gx = _sum_rows(g_rows, rev, torch.ones_like(g_rows[:, 0]), case["T"])
        gg = torch.empty(order.numel(), dtype=torch.float64, device=x.device)
        gg[order] = g_gates.double()
        return [x.double()[rev], None, None, gates.double().reshape(-1)[order], None, None, gx,
                gg.view(gates.shape)]
    if kind == "layer":
        x, go, weights = _layer_inputs(case, seed)
        T, D, k, E = case["T"], case["D"], case["k"], case["E"]
        # the layer's own choice of experts, made from its bf16 logits
        ids = torch.topk(torch.nn.functional.linear(x.view(T, D), weights[0]), k, dim=-1).indices
        x64 = x.double().requires_grad_(True)
        ws = [v.double().requires_grad_(True) for v in weights]
        flat = x64.view(T, D)
        gates = torch.softmax((flat @ ws[0].t()).gather(1, ids), dim=-1)
        out = torch.zeros(T, D, dtype=torch.float64, device=x.device)
        for e in range(E):
            t, j = (ids == e).nonzero(as_tuple=True)
            h = torch.nn.functional.gelu(flat[t] @ ws[1 + 2 * e].t()) @ ws[2 + 2 * e].t()
            out = out.index_add(0, t, h * gates[t, j][:, None])
        grads = torch.autograd.grad(out.view_as(x64), [x64, *ws], go.double())
        return [out.detach().view_as(x64), *grads]
    x, idx, w = _reduce_inputs(case, seed)
    return _sum_rows(x, idx, w, case["T"])
