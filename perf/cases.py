"""The work whose speed is watched: what a user of this framework has it do, through its public entry points.

Four kinds of work, each over the sizes it is met with:

  path    the execution path of a run, prepared once per graph and train mask: forward groups, mask chain,
          compaction, group split, execution plans (``workload.prepare``)
  epoch   one training epoch of a whole model: forward, loss, pruned backward, Adam step (``train.Trainer``)
  layer   forward and backward of one graph convolution (``gcn_conv.GCNConv`` under autograd)
  agg     the aggregations of one epoch alone, forward and pruned backward, for a caller that does its own dense
          algebra (the C ABI through ``capi``; the plans and workspaces are the caller's)

Graphs: uniform random, Chung-Lu power law (any vertex count) and R-MAT (a power of two), all symmetric with
self-loops; the train mask is Bernoulli.  Everything is fp32 with int32 indices, the framework's only types.
"""
import math

import torch

from eppgcn_amd import capi, graphs, train, workload
from eppgcn_amd.gcn_conv import GCNConv
from eppgcn_amd.param import backInputProperty, inputProperty, maskInputProperty

FEATURES, CLASSES = 96, 22      # input width and class count of the repository's own model


def listed():
    return [
        # the smallest graph that citation-network models are trained on: the epoch is host work and launches
        {"name": "epoch_uniform_2708", "kind": "epoch", "graph": "uniform", "n": 2708, "pairs": 1.95, "ratio": 0.1,
         "layers": 2, "features": FEATURES, "hidden": 16, "classes": CLASSES},
        # a medium power-law graph, the same model
        {"name": "epoch_chunglu_19717", "kind": "epoch", "graph": "chunglu", "n": 19717, "pairs": 2.25, "ratio": 0.1,
         "layers": 2, "features": FEATURES, "hidden": 16, "classes": CLASSES},
        # a deeper and wider model on it (the depth sweep trains 3 to 6 layers); larger graphs are taken layer by layer
        {"name": "epoch_chunglu_19717_deep", "kind": "epoch", "graph": "chunglu", "n": 19717, "pairs": 2.25,
         "ratio": 0.3, "layers": 4, "features": FEATURES, "hidden": 32, "classes": CLASSES},
        # the input layer of the model on a million vertices: its backward path is the one-hop closure of the mask
        {"name": "layer_rmat20_96x16", "kind": "layer", "graph": "rmat", "n": 1 << 20, "pairs": 4, "ratio": 0.1,
         "hops": 1, "in_dim": FEATURES, "out_dim": 16, "hidden_layer": False},
        # the output layer on four million vertices: activation of its input fused, gradient to the layer below
        {"name": "layer_rmat22_16x22", "kind": "layer", "graph": "rmat", "n": 1 << 22, "pairs": 16, "ratio": 0.1,
         "hops": 0, "in_dim": 16, "out_dim": CLASSES, "hidden_layer": True},
        # the benchmark's epoch of aggregations: widths 16 and 22, forward and pruned backward
        {"name": "agg_rmat22_16_22", "kind": "agg", "graph": "rmat", "n": 1 << 22, "pairs": 16, "ratio": 0.1,
         "layers": 2, "hidden": 16, "classes": CLASSES},
        # wide hidden layers on a million vertices, a sparse mask and a dense one
        {"name": "agg_rmat20_64", "kind": "agg", "graph": "rmat", "n": 1 << 20, "pairs": 4, "ratio": 0.01,
         "layers": 1, "hidden": 64, "classes": 64},
        {"name": "agg_rmat20_256", "kind": "agg", "graph": "rmat", "n": 1 << 20, "pairs": 4, "ratio": 0.5,
         "layers": 1, "hidden": 256, "classes": 256},
        # sizes that fit no tile: odd vertex count, odd width
        {"name": "agg_chunglu_200003_47", "kind": "agg", "graph": "chunglu", "n": 200003, "pairs": 6.5, "ratio": 0.1,
         "layers": 1, "hidden": 47, "classes": 47},
        # path preparation, from a graph where it is launches and read-backs to one where it is memory traffic
        {"name": "path_chunglu_19717", "kind": "path", "graph": "chunglu", "n": 19717, "pairs": 2.25, "ratio": 0.1,
         "layers": 2, "hidden": 16, "classes": CLASSES},
        {"name": "path_rmat20", "kind": "path", "graph": "rmat", "n": 1 << 20, "pairs": 4, "ratio": 0.1,
         "layers": 2, "hidden": 16, "classes": CLASSES},
        {"name": "path_rmat22", "kind": "path", "graph": "rmat", "n": 1 << 22, "pairs": 16, "ratio": 0.1,
         "layers": 2, "hidden": 16, "classes": CLASSES},
    ]


def draw(rng):
    def spread(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    kind = rng.choice(["epoch", "layer", "agg", "path"])
    if kind == "epoch":
        n = int(spread(1000, 24000))
        graph = rng.choice(["uniform", "chunglu"])
    else:
        graph = rng.choice(["rmat", "chunglu"])
        n = 1 << rng.randint(16, 21) if graph == "rmat" else int(spread(20000, 1500000))
    pairs = float(rng.randint(3, 16)) if graph == "rmat" else round(spread(1.5, 9.0), 2)
    case = {"kind": kind, "graph": graph, "n": n, "pairs": pairs, "ratio": round(spread(0.01, 0.6), 3)}
    if kind == "layer":
        hidden_layer = rng.random() < 0.5
        case.update(hops=rng.randint(0, 1), in_dim=rng.randint(8, 64) if hidden_layer else rng.randint(16, 200),
                    out_dim=rng.randint(7, 64), hidden_layer=hidden_layer)
    elif kind == "agg":
        # the gathered volume stays below that of the widest listed case
        widest = max(24, min(256, int(1.5e9 / (n * (1 + 2 * pairs)) / 2)))
        case.update(layers=rng.randint(1, 2), hidden=int(spread(12, widest)), classes=int(spread(7, min(64, widest))))
    else:
        layers = rng.randint(2, 5)
        case.update(layers=layers, hidden=rng.randint(8, 32), classes=rng.randint(3, 32))
        if kind == "epoch":
            case.update(features=rng.randint(32, 200))
    return case


# ---------------------------------------------------------------- inputs
def _graph(case, seed, dev):
    n = int(case["n"])
    if case["graph"] == "rmat":
        return graphs.rmat_graph(n.bit_length() - 1, int(case["pairs"]), seed=seed, device=dev)
    make = graphs.uniform_graph if case["graph"] == "uniform" else graphs.chung_lu_graph
    return make(n, int(n * case["pairs"]), seed=seed, device=dev)


def _closure(g, mask):
    """The vertices whose features a layer above needs when `mask` are its targets: the mask and its neighbours."""
    near = mask.clone()
    near[g.column_index[mask[g.row_index()]].long()] = True
    return near


def _widths(case):
    return [case["hidden"]] * (case["layers"] - 1) + [case["classes"]]


def prepare(case, seed):
    dev = torch.device("cuda:0")
    kind = case["kind"]
    # a run's graph is the dataset's and its train mask is drawn anew: the sizes of a prepared path follow the graph
    g = _graph(case, 0 if kind == "path" else seed, dev)
    mask = graphs.bernoulli_mask(g.num_nodes, case["ratio"], seed + 1, dev)
    if kind == "path":
        return {"kind": kind, "graph": g, "mask": mask, "layers": case["layers"], "widths": _widths(case)}
    if kind == "epoch":
        ds = train.GraphDataset(g, case["features"], case["classes"], case["layers"], train_mask=mask,
                                labels="uniform", feature_seed=seed + 2, label_seed=seed + 3)
        tr = train.Trainer(g, hidden=case["hidden"], weight_seed=seed + 4, dataset=ds)
        tr.train_step(True, phase_timers=False)          # the first iteration prepares the execution path
        return {"kind": kind, "trainer": tr}
    if kind == "layer":
        return _prepare_layer(case, seed, g, mask)
    # agg: plans and workspaces belong to the caller, one workspace per layer, shared by its two calls
    n, widths = g.num_nodes, _widths(case)
    wl = workload.prepare(g, case["layers"], train_mask=mask, widths=tuple(widths))
    layers = []
    for k, width in enumerate(widths):
        path = wl.paths[k]
        reach = mask if k == len(widths) - 1 else wl.ngh_masks[len(widths) - 2 - k]
        x = graphs.normal32(seed + 5 + k, (n, width), dev)
        dy = graphs.normal32(seed + 5 + k, (n, width), dev, 1) * reach[:, None]
        ws = capi.feature_workspace(n, width, dev, [wl.plans.get(width), path.plan])
        layers.append({"x": x, "dy": dy, "path": path, "plan": wl.plans.get(width), "ws": ws,
                       "y": torch.empty_like(x), "dx": torch.empty_like(x)})
    return {"kind": kind, "graph": g, "wl": wl, "layers": layers}


def _prepare_layer(case, seed, g, mask):
    """One convolution with its forward groups and its compacted backward path, as the training driver wires them."""
    n, e, dev = g.num_nodes, g.num_edges, mask.device
    reach = _closure(g, mask) if case["hops"] else mask

    class Info:
        num_nodes, num_features, avg_degree, avg_edgeSpan = n, case["in_dim"], g.avg_degree, -1

    info = inputProperty(g.row_pointers, g.column_index, g.degrees, 32, 32, 8, 100, hiddenDim=case["out_dim"],
                         dataset_obj=Info(), manual_mode=False)
    info.decider()
    ops = train.gnnadvisor()
    info.partPtr, info.part2Node = ops.build_part(info.partSize, g.row_pointers)
    edge_mask = torch.full((e,), -1, dtype=torch.int32, device=dev)
    degs = torch.zeros(n, dtype=torch.int32, device=dev)
    marking = maskInputProperty(reach, torch.zeros(0, dtype=torch.bool, device=dev), edge_mask, degs, 1, 1,
                                case["out_dim"])
    back = backInputProperty(degrees=g.degrees, dim=case["out_dim"], layer=1)
    conv = GCNConv(case["in_dim"], case["out_dim"], relu_input=case["hidden_layer"]).to(dev)
    with torch.no_grad():
        conv.weights.copy_(graphs.uniform_weights(seed + 4, case["in_dim"], case["out_dim"], dev))
    x = graphs.normal32(seed + 2, (n, case["in_dim"]), dev).requires_grad_(case["hidden_layer"])
    dy = graphs.normal32(seed + 3, (n, case["out_dim"]), dev) * reach[:, None]
    info.set_hidden() if case["hidden_layer"] else info.set_input()
    with torch.no_grad():
        conv(x, info, marking, back, True, False)        # the first iteration marks the path
    ids, edge_list, found = ops.compact_back_edge(edge_mask, g.column_index)
    part_pointer, parts = ops.split_back_part(degs, e, 32)
    back.fillProperty(ids, part_pointer, edge_list, 32, int(parts[0].item()))
    marking.backEdgeMask = None
    return {"kind": "layer", "conv": conv, "x": x, "dy": dy, "info": info, "marking": marking, "back": back}


# ---------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind == "path":
        wl = workload.prepare(state["graph"], state["layers"], train_mask=state["mask"], widths=tuple(state["widths"]))
        out = {"part_ptr": wl.part_ptr, "part2node": wl.part2node, "masks": wl.ngh_masks, "size": wl.part_size}
        for p in wl.paths:
            out["path%d" % p.layer] = {"ids": p.ids, "edge_list": p.edge_list, "part_pointer": p.part_pointer,
                                       "node_degs": p.node_degs, "groups": p.num_parts, "edges": p.valid_len,
                                       "nodes": p.valid_node, "gathered": p.gathered_rows}
        return out
    if kind == "epoch":
        tr = state["trainer"]
        loss = tr.train_step(False, phase_timers=False)
        weights = list(tr.model.parameters())
        return {"loss": loss, "grads": [w.grad for w in weights], "weights": weights}
    if kind == "layer":
        conv, x = state["conv"], state["x"]
        y = conv(x, state["info"], state["marking"], state["back"], False, False)
        wrt = [conv.weights] + ([x] if x.requires_grad else [])
        return {"y": y, "grads": list(torch.autograd.grad(y, wrt, state["dy"]))}
    g, wl = state["graph"], state["wl"]
    for s in state["layers"]:
        capi.spmm_forward(s["x"], g.column_index, g.degrees, wl.part_ptr, wl.part2node, wl.part_size,
                          row_pointers=g.row_pointers, out=s["y"], workspace=s["ws"], plan=s["plan"])
    for k in reversed(range(len(state["layers"]))):
        s = state["layers"][k]
        p = s["path"]
        capi.ours_backward(s["dy"], p.ids, p.part_pointer, p.edge_list, g.degrees, p.num_parts, p.part_size, p.layer,
                           out=s["dx"], workspace=s["ws"], plan=p.plan, gathered_rows=p.gathered_rows)
    return {"y": [s["y"] for s in state["layers"]], "dx": [s["dx"] for s in state["layers"]]}


# ---------------------------------------------------------------- what a pass cannot do without
def _sizes(case):
    """(vertices, expected CSR slots).  R-MAT pairs repeat: the share of distinct ones was fitted to graphs of scale
    12 to 22 with 4 to 16 pairs per vertex (within 1 %)."""
    n, pairs = case["n"], case["pairs"]
    distinct = 1.0
    if case["graph"] == "rmat":
        distinct -= 0.0565 * (pairs / 4.0) ** 0.63 * 2.0 ** (-0.28 * (n.bit_length() - 17))
    return n, n * (1.0 + 2.0 * pairs * distinct)


def _reached(case, hops):
    """Expected share of the vertices within `hops` of the mask, for vertices of average degree."""
    share = case["ratio"]
    for _ in range(hops):
        share = 1.0 - (1.0 - share) ** (1.0 + 2.0 * case["pairs"])
    return share


def work(case):
    n, e = _sizes(case)
    kind = case["kind"]
    csr = 4.0 * e + 8.0 * n                              # column ids, row pointers, scale vector: once per pass
    if kind == "layer":
        k, d = case["in_dim"], case["out_dim"]
        kept = e * _reached(case, case["hops"])
        dx = 4.0 * n * k if case["hidden_layer"] else 0.0
        return {"bytes": csr + 4.0 * kept + 4.0 * n * (2 * k + 2 * d) + dx,
                "flops": 2.0 * (e + kept) * d + 2.0 * n * k * d * (3 if case["hidden_layer"] else 2)}
    layers = case["layers"]
    kept = [e * _reached(case, layers - 1 - k) for k in range(layers)]
    if kind == "path":
        # the mask decides every slot; per layer three arrays of e + 1 words (zero behind the kept slots), the kept
        # degrees and the neighbour mask come out, and the groups of the forward direction
        return {"bytes": layers * (4.0 * e + 12.0 * e + 4.0 * n + 2.0 * n) + 4.0 * n + 8.0 * e / 16.0,
                "flops": layers * e}
    widths = _widths(case)
    if kind == "agg":
        return {"bytes": csr + sum(4.0 * v for v in kept) + sum(16.0 * n * d for d in widths),
                "flops": sum(2.0 * (e + v) * d for v, d in zip(kept, widths))}
    fan_in = [case["features"]] + widths[:-1]
    flops = sum(2.0 * (e + v) * d + 2.0 * n * k * d * (2 if i == 0 else 3)
                for i, (v, d, k) in enumerate(zip(kept, widths, fan_in)))
    # every layer's input is read in both directions, its output and the gradients are written and read once
    words = sum(2.0 * n * (k + d) + (0 if i == 0 else n * k) for i, (d, k) in enumerate(zip(widths, fan_in)))
    return {"bytes": csr + sum(4.0 * v for v in kept) + 4.0 * words, "flops": flops}


def tolerance(case):
    # Measured against the same pass with its sums in another order (no execution plans, library matrix products):
    # aggregations rel 1.6e-8, max 5e-7; with weight gradients (sums over all vertices) rel 3e-6, max 1.3e-5.  An
    # aggregation that applies the two scale factors in another order rounds every term once more (up to 1e-7).
    if case["kind"] == "path":
        return "exact"
    if case["kind"] == "agg":
        return {"rel": 5e-7, "max": 5e-6}
    return {"rel": 1.2e-5, "max": 6e-5}
