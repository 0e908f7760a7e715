"""Performance cases of the routing and expert path, through the public entry points.

A case is one pass of a program that uses this framework for inference: a routed layer
(scatter router -> expert FFN in two grouped GEMMs -> gather router), a route without experts, the
routing ops on their own, or a grouped FFN over given loads.  ``listed`` holds the sizes of the
repository's configurations, tests and benchmark (and of decode batches); ``draw`` gives more of the
same ranges: 8 to 131072 cells of 8 to 2048 elements, 2 to 128 paths, one or two paths per cell,
fp32 / fp16 / bf16, odd and ragged sizes among them.
"""
import math

import torch
import torch.nn as nn

import brt
import brt._C.router as c_router
from brt.jit import make_jit_kernel
from brt.router import GatherRouter, ScatterRouter, SwinMoEScatterRouter

_DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}

# How a program builds its fused dispatch fabric: as the reference's programs do, or with the
# switches that keep a layer free of host reads, of the dispatch, or of the dense route.
_FORMS = {
    "drop_in": {},
    "static_rows": {"static_rows": True},
    "defer": {"defer_dispatch": True},
    "compact": {"compact_route": True},
    "compact_defer": {"compact_route": True, "defer_dispatch": True},
    # ... and the expert's last kernel is handed the residual (one path per cell only)
    "folded": {"compact_route": True, "defer_dispatch": True},
}


def _layer(name, tokens, d, d_ff, experts, top_k, form, dtype="bf16", capacity_factor=1.25, skew=0.0, bias=False):
    return {"name": name, "kind": "layer", "tokens": tokens, "d": d, "d_ff": d_ff, "experts": experts, "top_k": top_k,
            "form": form, "dtype": dtype, "capacity_factor": capacity_factor, "skew": skew, "bias": bias}


def listed():
    return [
        # decode steps of a serving batch: few cells, every expert that gets one streams its weights
        _layer("decode_24_tokens", 24, 768, 3072, 8, 1, "compact_defer"),
        _layer("decode_96_tokens_top2", 96, 1024, 4096, 32, 2, "compact", capacity_factor=2.0),
        # a program of the reference as it stands: fp32 activations and parameters, no switches set
        _layer("switch_1k_fp32_drop_in", 1024, 512, 2048, 16, 1, "drop_in", dtype="fp32"),
        # the benchmark's Switch layer (8192 tokens, 64 experts, capacity 160)
        _layer("switch_8k", 8192, 768, 3072, 64, 1, "static_rows"),
        # the same layer on a ragged batch, with everything folded into the expert kernels
        _layer("switch_5003_folded", 5003, 768, 3072, 64, 1, "folded"),
        # a large prefill batch: thousands of rows per expert
        _layer("prefill_32k", 32768, 1024, 4096, 16, 1, "compact_defer"),
        # top-2 with skewed loads and a gate-weighted combine
        _layer("top2_16k_skewed", 16384, 1024, 4096, 32, 2, "compact", capacity_factor=2.0, skew=1.2),
        # task-MoE: one grouped FFN over ragged loads (most experts light, a few with thousands of rows)
        {"name": "task_ffn_128e", "kind": "ffn", "rows": 32768, "d": 2048, "d_ff": 8192, "experts": 128, "alpha": 0.3,
         "bias": False},
        # Swin-MoE routing: many short rows, capacity-padded with a fixed stride per path
        {"name": "swin_100352", "kind": "swin", "tokens": 100352, "d": 96, "experts": 8, "dtype": "fp16",
         "capacity_factor": 1.0},
        # routing alone through the fused routers, identity experts (1024 x 512, 16 paths)
        {"name": "route_1k_fp32", "kind": "route", "tokens": 1024, "d": 512, "experts": 16, "top_k": 1, "form": "drop_in",
         "dtype": "fp32"},
        # the ops themselves: throttle, index generation, dispatch, gate-weighted combine into fp32
        {"name": "ops_16k_top2", "kind": "ops", "tokens": 16384, "d": 1024, "experts": 32, "top_k": 2, "dtype": "bf16",
         "skew": 1.2},
        # the default routers (one flow per path, cells found again by their tags), as dynamic CNNs use them
        {"name": "branches_2k_fp32", "kind": "branches", "tokens": 2048, "d": 512, "experts": 4, "top_k": 2,
         "dtype": "fp32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A feature width the expert kernels take: mostly whole K-steps of 64, some multiples of 8."""
    unit = 64 if rng.random() < 0.75 else 8
    return max(lo, _log_int(rng, lo, hi) // unit * unit)


def draw(rng):
    kind = rng.choice(["layer"] * 6 + ["ffn", "swin", "route", "route", "ops", "branches"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if kind == "layer":
        d = _width(rng, 256, 2048)
        d_ff = d * rng.choice([2, 4]) if rng.random() < 0.8 else _width(rng, d, 4 * d)
        top_k = rng.choice([1, 1, 2])
        most = int(min(32768, 2.0e12 / (4.0 * d * d_ff * top_k)))  # no dearer than the largest listed case
        fp32 = rng.random() < 0.2
        forms = ["drop_in", "static_rows", "defer", "compact_defer"] + ([] if fp32 else ["folded"])
        form = rng.choice(forms if top_k == 1 else ["drop_in", "compact", "compact_defer"])
        experts = rng.choice([e for e in (4, 8, 12, 16, 32, 64, 128) if 2 * e * d * d_ff * (4 if fp32 else 2) <= 8.6e9])
        return _layer(None, _log_int(rng, 8, most), d, d_ff, experts, top_k, form,
                      dtype="fp32" if fp32 else "bf16", capacity_factor=rng.choice([1.25, 2.0]),
                      skew=rng.choice([0.0, 0.0, 1.2]), bias=rng.random() < 0.25)
    if kind == "ffn":
        d = _width(rng, 256, 2048)
        d_ff = 4 * d if rng.random() < 0.8 else _width(rng, d, 4 * d)
        most = int(min(32768, 2.0e12 / (4.0 * d * d_ff)))
        return {"kind": kind, "rows": _log_int(rng, 16, most), "d": d, "d_ff": d_ff,
                "experts": rng.choice([4, 8, 16, 60, 128]), "alpha": rng.choice([0.3, 1.0, 100.0]),
                "bias": rng.random() < 0.5}
    tokens = _log_int(rng, 8, 131072)
    # any width, also rows that are not whole 16-byte units
    d = _log_int(rng, 8, 2048)
    d = d if rng.random() < 0.25 else max(8, d // 8 * 8)
    tokens = max(8, min(tokens, (1 << 26) // d))  # at most 256 MB of fp32 rows
    if kind == "swin":
        return {"kind": kind, "tokens": tokens, "d": d, "experts": rng.choice([4, 8, 16, 32]), "dtype": dtype,
                "capacity_factor": rng.choice([1.0, 1.25])}
    if kind == "route":
        top_k = rng.choice([1, 1, 2])
        return {"kind": kind, "tokens": tokens, "d": d, "experts": rng.choice([4, 8, 12, 16, 64, 128]), "top_k": top_k,
                "form": rng.choice(["drop_in", "static_rows", "compact"] if top_k == 1 else ["drop_in", "compact"]),
                "dtype": dtype}
    if kind == "ops":
        return {"kind": kind, "tokens": tokens, "d": d, "experts": rng.choice([8, 16, 32, 64]), "top_k": rng.choice([1, 2, 4]),
                "dtype": dtype, "skew": rng.choice([0.0, 1.2])}
    return {"kind": kind, "tokens": min(tokens, 16384), "d": d, "experts": rng.choice([2, 4, 8]), "top_k": rng.choice([1, 2]),
            "dtype": dtype}


# ------------------------------------------------------------------------------------ inputs
def _scores(gen, cells, paths, skew):
    """Router probabilities of N(0,1) logits; ``skew`` > 0 adds the log of a Zipf(skew) pmf over the
    paths in random order, so that a few paths are popular."""
    logits = torch.randn(cells, paths, device="cuda", generator=gen)
    if skew > 0:
        pmf = 1.0 / torch.arange(1, paths + 1, device="cuda", dtype=torch.float32) ** skew
        logits += torch.log(pmf / pmf.sum())[torch.randperm(paths, device="cuda", generator=gen)]
    return torch.softmax(logits, dim=1)


def _normal(gen, *shape, dtype, scale=1.0):
    return torch.randn(*shape, device="cuda", generator=gen, dtype=torch.float32 if dtype != torch.bfloat16 else dtype
                       ).mul_(scale).to(dtype)


def _experts(gen, count, d_in, d_out, dtype, bias, activation):
    """``count`` Linear branches with N(0, 0.02) weights, the fused kernel over them and the
    parameter list it is called with."""
    weight = _normal(gen, count, d_out, d_in, dtype=dtype, scale=0.02)
    offset = _normal(gen, count, d_out, dtype=dtype, scale=0.02) if bias else None
    branches = nn.ModuleList(nn.Linear(d_in, d_out, bias=bias, device="meta") for _ in range(count))
    operands = []
    for e, branch in enumerate(branches):
        branch.weight = nn.Parameter(weight[e], requires_grad=False)
        operands.append(branch.weight)
        if bias:
            branch.bias = nn.Parameter(offset[e], requires_grad=False)
            operands.append(branch.bias)
    return make_jit_kernel(branches, None, opt_level="homo_fuse", activation=activation), operands


def _capacity(case):
    per_path = -(-case["tokens"] // case["experts"])
    return max(4, case["top_k"] * int(case["capacity_factor"] * per_path))


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case, "annotate": brt.Annotator([0])}
    kind = case["kind"]
    if kind == "ffn":
        rows, experts = case["rows"], case["experts"]
        share = torch._standard_gamma(torch.full((experts,), case["alpha"], dtype=torch.float64),
                                      generator=torch.Generator().manual_seed(seed))
        share = share / share.sum() * rows
        loads = share.floor().to(torch.int64)
        order = torch.argsort(loads - share)  # largest remainder first: the loads add up to the rows
        loads[order[:rows - int(loads.sum())]] += 1
        state["loads"] = loads.to(torch.int32).cuda()
        state["x"] = _normal(gen, rows, case["d"], dtype=torch.bfloat16)
        state["wi"], state["wi_operands"] = _experts(gen, experts, case["d"], case["d_ff"], torch.bfloat16, case["bias"], "gelu")
        state["wo"], state["wo_operands"] = _experts(gen, experts, case["d_ff"], case["d"], torch.bfloat16, case["bias"], None)
        return state
    dtype = _DTYPES[case["dtype"]]
    tokens, d, experts = case["tokens"], case["d"], case["experts"]
    state["x"] = _normal(gen, tokens, d, dtype=dtype)
    state["score"] = _scores(gen, tokens, experts, case.get("skew", 0.0))
    if kind in ("layer", "route"):
        fabric = dict(_FORMS[case["form"]])
        if kind == "layer":
            fabric["supported_capacities"] = _capacity(case)
        weighted = case["top_k"] > 1
        state["scatter"] = ScatterRouter(protocol_type="topk", protocol_kwargs={"top_k": case["top_k"]},
                                         fabric_type="fused_dispatch", fabric_kwargs=fabric).cuda()
        state["gather"] = GatherRouter(fabric_type="fused_combine", fabric_kwargs={"transform": weighted}).cuda()
        # with one path per cell the layer's output starts as the hidden states (cells over capacity keep theirs)
        state["residual"] = None if weighted or kind == "route" else state["x"].clone()
        if kind == "layer":
            state["wi"], state["wi_operands"] = _experts(gen, experts, d, case["d_ff"], dtype, case["bias"], "gelu")
            state["wo"], state["wo_operands"] = _experts(gen, experts, case["d_ff"], d, dtype, case["bias"], None)
    elif kind == "swin":
        state["scatter"] = SwinMoEScatterRouter(
            protocol_kwargs={"top_k": 1, "capacity_factor": case["capacity_factor"]}, fabric_type="fused_dispatch",
            fabric_kwargs={"capacity_padding": True, "max_path_padding": True}).cuda()
        state["gather"] = GatherRouter(fabric_type="fused_combine", fabric_kwargs={"max_path_padding": True}).cuda()
    elif kind == "ops":
        top = torch.topk(state["score"], case["top_k"], dim=1).indices
        state["mask"] = torch.zeros(tokens, experts, dtype=torch.int32, device="cuda").scatter_(1, top, 1)
        gates = state["score"] * state["mask"]
        state["gates"] = gates / gates.sum(dim=1, keepdim=True)
        per_path = -(-tokens // experts)
        state["threshold"] = torch.full((experts,), case["top_k"] * 2 * per_path, dtype=torch.int32, device="cuda")
    else:
        state["scatter"] = ScatterRouter(protocol_type="topk", protocol_kwargs={"top_k": case["top_k"]}).cuda()
        state["gather"] = GatherRouter().cuda()
    return state


# -------------------------------------------------------------------------------------- passes
def _run_ffn(state, x, loads):
    case = state["case"]
    hidden = torch.empty(x.shape[0], case["d_ff"], dtype=x.dtype, device=x.device)
    state["wi"](shared_inputs=[x, hidden], standalone_inputs=state["wi_operands"], capacities=loads)
    out = torch.empty(x.shape[0], case["d"], dtype=x.dtype, device=x.device)
    folded = {"residual": state["residual"]} if case.get("form") == "folded" else {}
    state["wo"](shared_inputs=[hidden, out], standalone_inputs=state["wo_operands"], capacities=loads, **folded)
    return out


def _run_layer(state):
    routed = state["scatter"](state["annotate"](state["x"]), state["score"])
    rows, tags, loads, extra = brt.to_torch_tensor(routed, retrieve_attr=True)
    layer_loads = loads[-1]
    y = _run_ffn(state, rows, layer_loads)
    out = state["gather"](brt.to_grid_tensor(y, tags, loads, extra), state["residual"], state["score"])
    return {"out": brt.to_torch_tensor(out), "loads": layer_loads}


def _run_route(state):
    routed = state["scatter"](state["annotate"](state["x"]), state["score"])
    loads = routed.load
    rows = brt.to_torch_tensor(routed)
    out = state["gather"](routed, None, state["score"])
    return {"rows": rows, "loads": loads, "out": brt.to_torch_tensor(out)}


def _run_swin(state):
    routed, _ = state["scatter"](state["annotate"](state["x"]), state["score"], None, None)
    loads = routed.load
    rows = brt.to_torch_tensor(routed)
    out = state["gather"](routed)
    return {"rows": rows, "loads": loads, "out": brt.to_torch_tensor(out)}


def _run_ops(state):
    taken = torch.zeros_like(state["threshold"])
    mask, taken = c_router.throttle_hotmask(state["mask"], taken, state["threshold"])
    route = c_router.generate_route(mask)
    (rows,) = c_router.dispatch_with_indices_and_loads(state["x"], route.indices, route.loads, route=route)
    (out,) = c_router.combine_with_indices_and_loads(rows, route.indices, route.loads, state["gates"],
                                                     out_dtype=torch.float32, route=route)
    return {"indices": route.indices, "loads": route.loads, "taken": taken, "out": out}


def _run_branches(state):
    flows = state["scatter"](state["annotate"](state["x"]), state["score"])
    return {"out": brt.to_torch_tensor(state["gather"](flows))}


def run(state):
    kind = state["case"]["kind"]
    if kind == "layer":
        return _run_layer(state)
    if kind == "ffn":
        return _run_ffn(state, state["x"], state["loads"])
    return {"route": _run_route, "swin": _run_swin, "ops": _run_ops, "branches": _run_branches}[kind](state)


# ------------------------------------------------------------------------- work and tolerances
def _kept(case, capacity):
    """Expected (cell, path) pairs a capacity leaves and paths that get any, by the share of every path under the skew."""
    entries = case["tokens"] * case["top_k"]
    shares = [1.0 / (e + 1) ** case["skew"] for e in range(case["experts"])]
    shares = [s / sum(shares) for s in shares]
    return sum(min(capacity, entries * s) for s in shares), sum(1.0 - (1.0 - s) ** entries for s in shares)


def work(case):
    kind = case["kind"]
    size = 2 if kind == "ffn" else _DTYPES[case["dtype"]].itemsize
    d, experts = case["d"], case["experts"]
    if kind == "ffn":
        rows = case["rows"]
        used = min(experts, rows) * (0.85 if case["alpha"] < 0.5 else 1.0)  # light experts draw no row at all
        weights = 2 * used * d * case["d_ff"] * size
        return {"bytes": weights + 2 * rows * (d + case["d_ff"]) * size, "flops": 4.0 * rows * d * case["d_ff"]}
    tokens = case["tokens"]
    entries = tokens * case.get("top_k", 1)
    score = 4 * tokens * experts
    if kind == "layer":
        rows, used = _kept(case, _capacity(case))
        weights = 2 * used * d * case["d_ff"] * size
        return {"bytes": score + weights + (tokens * d + 2 * rows * case["d_ff"] + tokens * d) * size,
                "flops": 4.0 * rows * d * case["d_ff"]}
    if kind == "ops":
        # mask in, index matrix and gates, the cells in, the rows out and in again, the fp32 result out
        rows, _ = _kept(case, case["top_k"] * 2 * -(-tokens // experts))
        return {"bytes": 3 * score + (min(tokens, rows) + 2 * rows) * d * size + tokens * d * 4, "flops": 2.0 * rows * d}
    # the scores, the cells in, the rows out and in again, the result out
    return {"bytes": score + (2 * tokens + 2 * entries) * d * size, "flops": 0.0}


def tolerance(case):
    """Four times the distance from an evaluation in 64 bits that uses the same inputs."""
    kind = case["kind"]
    if kind in ("layer", "ffn"):
        # bf16 operands, the hidden state and the output rounded to bf16: 2.3e-3 (top-1) and 2.9e-3
        # (top-2, every row rounded before the sum) of the norm, 3.4e-3 where fp32 operands are rounded first;
        # the largest error 1.7e-2 of the rms, 2.8e-2 where the rows of popular experts are summed
        return {"rel": 1.2e-2, "max": 0.11 if case.get("top_k") == 2 else 0.07}
    if kind == "ops":  # products and sums of up to four terms in fp32: 2.9e-8, largest 1.1e-7
        return {"rel": 2e-7, "max": 1e-6}
    if kind == "route" and case["top_k"] > 1:  # an fp32 sum rounded to the data type (fp16: 2.1e-4, largest 4.9e-4)
        unit = {"fp32": 2.0 ** -24, "fp16": 2.0 ** -11, "bf16": 2.0 ** -8}[case["dtype"]]
        return {"rel": 1.7 * unit, "max": 4 * unit}
    return "exact"  # rows are moved, or a cell is added to itself
