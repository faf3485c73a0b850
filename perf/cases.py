"""What this framework is used for, as cases that can be timed: whole samplers (GraphSAGE in its
three calling styles, LADIES, GraphSAINT-style subgraphs, walks) and the operators that
samplers and models are written with (weighted sampling, edge features, edge-data
normalisation, loading an edge list), over synthetic R-MAT graphs (a=.57, b=.19, c=.19).

A case is a dict of plain values; `listed()` gives the fixed ones, `draw(rng)` one more of the
same ranges.  Every call that draws random numbers is given its seed first
(`gs.set_seed`), as a program that wants reproducible minibatches does.  How long a sampler's
outputs are depends on what it meets, so another input seed renumbers the nodes (or
reorders the edges) of a graph of the same shape: other inputs, outputs of the same length.
"""
import torch

import graph_sampling_amd as gs
from graph_sampling_amd import rmat

DEVICE = "cuda:0"


def listed():
    return [
        # one node-classification request of an online service: a few seeds, two small layers, on
        # a small graph; nothing but launches and latency
        {"name": "sage_online_32", "kind": "sage", "nodes": 1 << 17, "edges": 1 << 21, "seeds": 32,
         "fanouts": "10,5", "ids": 32, "weights": False, "replace": False},
        # the training minibatch of GraphSAGE on a paper-citation-sized graph with edge weights:
        # three layers in one call
        {"name": "sage_train_1024", "kind": "sage", "nodes": 111_000_000, "edges": 1_600_000_000,
         "seeds": 1024, "fanouts": "15,10,5", "ids": 32, "weights": True, "replace": False},
        # the same sampler written layer by layer (fused slice + sample, relabel) with the 64-bit
        # ids torch programs have by default, on a small dense social graph, with replacement
        {"name": "sage_layers_5000", "kind": "layers", "nodes": 233_000, "edges": 114_600_000,
         "seeds": 5000, "fanouts": "25,15", "ids": 64, "weights": False, "replace": True},
        # an epoch's worth of minibatches sampled 64 at a time: one sampling and one relabel call
        # per layer over all of them
        {"name": "super_batch_64x1024", "kind": "super", "nodes": 2_450_000, "edges": 124_000_000,
         "batches": 64, "seeds": 1024, "fanouts": "15,10,5", "ids": 32},
        # a LADIES minibatch (layer-wise importance sampling), compiled from the sampler as written
        {"name": "ladies_512", "kind": "ladies", "nodes": 2_450_000, "edges": 124_000_000,
         "seeds": 512, "picks": 512, "layers": 2, "ids": 32},
        # neighbours drawn by edge weight from the columns of a minibatch
        {"name": "weighted_5000x25", "kind": "weighted", "nodes": 233_000, "edges": 114_600_000,
         "seeds": 5000, "fanout": 25, "ids": 64, "replace": False},
        # random-walk corpus for skip-gram embeddings: a million walkers, eighty steps
        {"name": "walk_1m_80", "kind": "walk", "nodes": 4_000_000, "edges": 200_000_000,
         "walkers": 1_000_000, "length": 80, "ids": 32},
        # metapath walks over a heterogeneous graph of three relations
        {"name": "metapath_200k_30", "kind": "metapath", "nodes": 2_000_000, "edges": 50_000_000,
         "walkers": 200_000, "length": 30, "ids": 64},
        # GraphSAINT: the subgraph that the nodes of 2000 short walks induce, edge weights with it
        {"name": "saint_2000x4", "kind": "saint", "nodes": 233_000, "edges": 114_600_000,
         "seeds": 2000, "length": 4, "ids": 64, "weights": True},
        # attention scores: the dot product of both ends' features on every edge
        {"name": "dot_8m_64", "kind": "dot", "nodes": 2_450_000, "edges": 8_000_000, "heads": 1,
         "dim": 64, "ids": 32},
        # preparing the weights of a whole graph: squared column sums, columns scaled to one
        {"name": "normalize_124m", "kind": "normalize", "nodes": 2_450_000, "edges": 124_000_000,
         "axis": 0, "ids": 32},
        # an edge list with self loops, in no order, loaded and turned into the form samplers read
        {"name": "load_edges_14m", "kind": "load", "nodes": 2_450_000, "edges": 11_550_000,
         "to": "csc", "ids": 64},
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], spread evenly over its logarithm."""
    return min(hi, max(lo, int(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["sage", "sage", "layers", "super", "ladies", "weighted", "walk", "metapath",
                       "saint", "dot", "normalize", "load"])
    c = {"kind": kind, "ids": rng.choice([32, 64])}
    fanouts = lambda: rng.choice(["10,5", "25,10", "25,15", "5,5,5", "15,10,5", "7,3"])  # noqa: E731
    if kind == "sage":
        c["nodes"] = _between(rng, 1 << 14, 111_000_000)
        c["edges"] = min(1_600_000_000, c["nodes"] * _between(rng, 8, 50))
        c["seeds"] = _between(rng, 1, min(8192, c["nodes"]))
        c["fanouts"] = fanouts()
        c["weights"], c["replace"] = rng.random() < 0.5, rng.random() < 0.3
    elif kind == "layers":
        c["nodes"] = _between(rng, 1 << 14, 4_000_000)
        c["edges"] = min(124_000_000, c["nodes"] * _between(rng, 8, 492))
        c["seeds"] = _between(rng, 32, 5000)
        c["fanouts"] = fanouts()
        c["weights"], c["replace"] = rng.random() < 0.5, rng.random() < 0.5
    elif kind == "super":
        c["nodes"] = _between(rng, 1 << 17, 4_000_000)
        c["edges"] = min(124_000_000, c["nodes"] * _between(rng, 8, 50))
        c["batches"] = _between(rng, 4, 64)
        c["seeds"] = _between(rng, 64, 1024)
        c["fanouts"] = fanouts()
    elif kind == "ladies":
        c["nodes"] = _between(rng, 1 << 17, 2_450_000)
        c["edges"] = c["nodes"] * _between(rng, 8, 50)
        c["seeds"], c["picks"] = _between(rng, 64, 1000), _between(rng, 64, 2000)
        c["layers"] = 2
    elif kind == "weighted":
        c["nodes"] = _between(rng, 1 << 15, 2_450_000)
        c["edges"] = min(114_600_000, c["nodes"] * _between(rng, 8, 492))
        c["seeds"], c["fanout"] = _between(rng, 32, 5000), rng.randint(3, 25)
        c["replace"] = rng.random() < 0.4
    elif kind == "walk":
        c["nodes"] = _between(rng, 1 << 17, 4_000_000)
        c["edges"] = c["nodes"] * _between(rng, 8, 50)
        c["walkers"], c["length"] = _between(rng, 1000, 1_000_000), _between(rng, 4, 80)
    elif kind == "metapath":
        c["nodes"] = _between(rng, 1 << 17, 2_000_000)
        c["edges"] = c["nodes"] * _between(rng, 8, 25)
        c["walkers"], c["length"] = _between(rng, 1000, 1_000_000), _between(rng, 4, 30)
    elif kind == "saint":
        c["nodes"] = _between(rng, 1 << 17, 2_450_000)
        c["edges"] = min(114_600_000, c["nodes"] * _between(rng, 8, 492))
        c["seeds"], c["length"] = _between(rng, 200, 6000), rng.randint(2, 5)
        c["weights"] = rng.random() < 0.5
    elif kind == "dot":
        c["nodes"] = _between(rng, 1 << 15, 2_450_000)
        c["edges"] = _between(rng, 50_000, 8_000_000)
        c["heads"], c["dim"] = rng.choice([1, 1, 2, 4, 8]), rng.choice([8, 16, 32, 50, 64])
        if c["heads"] > 1:
            c["dim"] = min(c["dim"], 64 // c["heads"])
    elif kind == "normalize":
        c["axis"] = rng.choice([0, 0, 1])
        c["nodes"] = _between(rng, 1 << 15, 2_450_000)
        c["edges"] = min(124_000_000 if c["axis"] == 0 else 30_000_000,
                         c["nodes"] * _between(rng, 8, 50))
    else:
        c["nodes"] = _between(rng, 1 << 15, 2_450_000)
        c["edges"] = min(11_550_000, c["nodes"] * _between(rng, 4, 50))
        c["to"] = rng.choice(["csc", "csr"])
    return c


# ---------------------------------------------------------------------------------- inputs
def _id_type(case):
    return torch.int64 if case["ids"] == 64 else torch.int32


def _fanouts(case):
    return [int(k) for k in case["fanouts"].split(",")]


def _generator(seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    return gen


def _graph(case, seed):
    return rmat.rmat_csc(case["nodes"], case["edges"], seed=seed, device=DEVICE,
                         index_dtype=_id_type(case))


def _weights(case, gen):
    """(0, 1]: no edge is out of reach of a weighted sampler."""
    return 1.0 - torch.rand(case["edges"], generator=gen, device=DEVICE)


def _distinct(case, n, gen):
    """n node ids as an epoch's shuffled nodes give them; again from the start when it is over."""
    ids = torch.randperm(case["nodes"], generator=gen, device=DEVICE)[:n]
    while ids.numel() < n:
        ids = torch.cat([ids, ids])[:n]
    return ids


def _renumbered(case, seed, num_seeds, weights):
    """One graph and one set of seed nodes, node v called (v + shift) % nodes: the columns of the
    matrix move up by `shift`, those pushed out come first."""
    base = _generator(case["nodes"] % 1_000_003)
    indptr, indices = _graph(case, 0)
    data = _weights(case, base) if weights else None
    ids = _distinct(case, num_seeds, base)
    n = case["nodes"]
    shift = 1 + (seed * 2_654_435_761) % (n - 1)
    cut = int(indptr[n - shift])  # edges of the columns that stay in front of the cut
    length = indptr[1:] - indptr[:-1]
    torch.cumsum(torch.cat([length[n - shift:], length[:n - shift]]), 0, out=indptr[1:])
    indices = torch.cat([indices[cut:], indices[:cut]])
    indices += shift
    indices -= (indices >= n) * n
    if data is not None:
        data = torch.cat([data[cut:], data[:cut]])
    return gs.Matrix().load_csc(indptr, indices, data), ((ids + shift) % n).to(_id_type(case))


def _reordered(case, seed):
    """One weighted graph and one set of seed nodes, the edges of every column and the seeds in
    another order for every `seed` (a layer-wise sampler picks nodes by their number)."""
    base, gen = _generator(case["nodes"] % 1_000_003), _generator(seed)
    src, dst = rmat.rmat_edges(case["nodes"], case["edges"], seed=0, device=DEVICE)
    data = _weights(case, base)
    ids = _distinct(case, case["seeds"], base)
    order = torch.randperm(case["edges"], generator=gen, device=DEVICE)
    dst, perm = torch.sort(dst[order], stable=True)
    order = order[perm]
    indptr = torch.zeros(case["nodes"] + 1, dtype=torch.int64, device=DEVICE)
    torch.cumsum(torch.bincount(dst, minlength=case["nodes"]), 0, out=indptr[1:])
    A = gs.Matrix().load_csc(indptr, src[order].to(_id_type(case)), data[order])
    shuffled = ids[torch.randperm(case["seeds"], generator=gen, device=DEVICE)]
    return A, shuffled.to(_id_type(case))


def ladies(A, seeds, fanouts):
    """The sampler as its authors' example writes it against the matrix API."""
    blocks = []
    for fanout in fanouts:
        U = A[:, seeds]
        prob = U.sum(axis=1, powk=2)
        selected, _ = torch.ops.gs_ops.list_sampling_with_probs(U.row_ids(unique=False), prob,
                                                                fanout, False)
        nodes = torch.cat((seeds, selected)).unique()
        sub = U[nodes, :].divide(prob[nodes], axis=1).normalize(axis=0)
        seeds = sub.all_indices()
        blocks.insert(0, sub.to_dgl_block())
    return seeds, blocks


def prepare(case, seed):
    kind, gen = case["kind"], _generator(seed)
    s = {"case": case, "kind": kind, "draws": 7777}
    if kind in ("sage", "layers"):
        s["A"], s["seeds"] = _renumbered(case, seed, case["seeds"], case["weights"])
        s["fanouts"] = _fanouts(case)
    elif kind == "super":
        s["A"], s["seeds"] = _renumbered(case, seed, case["batches"] * case["seeds"], False)
        s["ptr"] = torch.arange(case["batches"] + 1, device=DEVICE) * case["seeds"]
        s["fanouts"] = _fanouts(case)
    elif kind == "ladies":
        s["A"], s["seeds"] = _reordered(case, seed)
        s["fanouts"] = [case["picks"]] * case["layers"]
        s["sampler"] = gs.jit.compile(ladies, (s["A"], s["seeds"], s["fanouts"]))
    elif kind == "weighted":
        s["A"], s["seeds"] = _renumbered(case, seed, case["seeds"], True)
    elif kind == "saint":
        s["A"], s["seeds"] = _renumbered(case, seed, case["seeds"], case["weights"])
    elif kind in ("walk", "metapath"):
        s["seeds"] = torch.randint(0, case["nodes"], (case["walkers"],), generator=gen,
                                   device=DEVICE).to(_id_type(case))
        if kind == "walk":
            s["A"] = gs.Matrix().load_csc(*_graph(case, seed))
        else:
            relations = [gs.Matrix().load_csc(*_graph(case, seed + 1_000_003 * r)) for r in range(3)]
            s["A"] = gs.HeteroMatrix()
            s["A"].load_from_homo(["paper", "author"],
                                  [("paper", "cites", "paper"), ("author", "writes", "paper"),
                                   ("paper", "written", "author")], relations)
            s["path"] = [("cites", "writes", "written", "writes")[i % 4]
                         for i in range(case["length"])]
    elif kind == "dot":
        s["A"] = gs.Matrix().load_csc(*_graph(case, seed))
        shape = (case["nodes"], case["dim"]) if case["heads"] == 1 else (
            case["nodes"], case["heads"], case["dim"])
        s["u"] = torch.rand(shape, generator=gen, device=DEVICE)
        s["v"] = torch.rand(shape, generator=gen, device=DEVICE)
    elif kind == "normalize":
        s["A"] = gs.Matrix().load_csc(*_graph(case, seed), _weights(case, gen))
    else:
        row, col = rmat.rmat_edges(case["nodes"], case["edges"], seed=seed, device=DEVICE)
        loops = torch.arange(case["nodes"], device=DEVICE)
        order = torch.randperm(case["edges"] + case["nodes"], generator=gen, device=DEVICE)
        s["row"] = torch.cat([row, loops])[order].to(_id_type(case))
        s["col"] = torch.cat([col, loops])[order].to(_id_type(case))
    return s


# ------------------------------------------------------------------------------- one pass
def _of_blocks(input_nodes, blocks):
    out = {"input_nodes": input_nodes}
    for i, b in enumerate(blocks):
        indptr, indices, order = b.csc() if b.format == "csc" else b.edges() + (None,)
        out["block%d" % i] = {"src": b.srcdata["_ID"], "indptr": indptr, "indices": indices,
                              "order": order, "e_ids": b.edata.get("_ID"), "w": b.edata.get("w")}
    return out


def run(s):
    kind, case = s["kind"], s["case"]
    gs.set_seed(s["draws"])
    if kind == "sage":
        return _of_blocks(*gs.sample_layers(s["A"], s["seeds"], s["fanouts"], case["replace"]))
    if kind == "layers":
        seeds, out = s["seeds"], []
        for k in s["fanouts"]:
            sub = s["A"]._graph._CAPI_FusedColumnwiseSlicingSampling(seeds, k, case["replace"])
            seeds, _, _, indptr, indices, _, _ = sub._CAPI_Relabel()
            data = sub._CAPI_GetData("default") if case["weights"] else None
            out.append((seeds, indptr, indices, data))
        return out
    if kind == "super":
        seeds, ptr, out = s["seeds"], s["ptr"], []
        for k in s["fanouts"]:
            sub = s["A"]._graph._CAPI_FusedColumnwiseSlicingSampling(seeds, k, False)
            indptr, indices, indices_ptr = sub._CAPI_GetBatchCSC(ptr)
            seeds, ptr, renamed, _ = torch.ops.gs_ops._CAPI_BatchCSRRelabel(seeds, ptr, indices,
                                                                            indices_ptr)
            out.append((seeds, ptr, indptr, renamed, indices_ptr))
        return out
    if kind == "ladies":
        return _of_blocks(*s["sampler"](s["A"], s["seeds"], s["fanouts"]))
    if kind == "weighted":
        U = s["A"][:, s["seeds"]]
        sub = U.columnwise_sampling(case["fanout"], case["replace"], U.get_data())
        block = sub.to_dgl_block()
        return _of_blocks(block.srcdata["_ID"], [block])
    if kind == "walk":
        return s["A"].random_walk(s["seeds"], case["length"])
    if kind == "metapath":
        return s["A"].metapath_random_walk_fused(s["seeds"], s["path"])
    if kind == "saint":
        trace = s["A"].random_walk(s["seeds"], case["length"]).reshape(-1)
        nodes = torch.ops.gs_ops._CAPI_Unique(trace[trace >= 0])  # (-1: the walk had ended)
        sub = s["A"]._graph._CAPI_FusionSlicing(nodes, nodes)
        return {"nodes": nodes, "csc": sub._CAPI_GetCSC()[:2],
                "w": sub._CAPI_GetData("default") if case["weights"] else None}
    if kind == "dot":
        return gs.ops.u_dot_v(s["A"], s["u"], s["v"])
    if kind == "normalize":
        return s["A"].sum(case["axis"], 2), s["A"].normalize(case["axis"]).get_data()
    A = gs.Matrix().load_coo(s["row"], s["col"])
    return A._graph._CAPI_GetCSC() if case["to"] == "csc" else A._graph._CAPI_GetCSR()


# ------------------------------------------------------------------ what it cannot do without
def _sampled(columns, degree, fanout):
    """Edges that sampling `fanout` from each of `columns` columns gives on a skewed graph: about
    two thirds of the places are filled at these degrees."""
    return columns * min(fanout, degree) * 0.66


def work(case):
    """Bytes: every input element that is used read once, every output element written once.
    How many edges a sampler meets depends on the graph; the numbers are estimates."""
    kind, b = case["kind"], case["ids"] // 8
    degree = case["edges"] / case["nodes"]
    if kind in ("sage", "layers", "super"):
        columns, total = float(case["seeds"] * case.get("batches", 1)), 0.0
        w = 8 if case.get("weights") else 0
        for k in _fanouts(case):
            edges = _sampled(columns, degree, k)
            frontier = min(columns + 0.7 * edges, float(case["nodes"]) * case.get("batches", 1))
            total += columns * (b + 24) + edges * (2 * b + w) + frontier * b
            columns = frontier
        return {"bytes": total, "flops": 0}
    if kind == "ladies":
        # the edges of the slice, weights with them, are looked at once; one probability per row
        edges = case["layers"] * (case["seeds"] + 0.5 * case["picks"]) * degree
        return {"bytes": edges * (b + 4) + case["layers"] * case["nodes"] * 8, "flops": 0}
    if kind == "weighted":
        edges = case["seeds"] * degree
        kept = case["seeds"] * min(case["fanout"], degree)
        return {"bytes": edges * 4 + kept * (3 * b + 8), "flops": 0}
    if kind in ("walk", "metapath"):
        # two offsets, a neighbour, a place of the trace; half of all walks end early
        return {"bytes": 0.5 * case["walkers"] * case["length"] * (16 + b)
                + case["walkers"] * (case["length"] + 1) * b, "flops": 0}
    if kind == "saint":
        nodes = min(case["seeds"] * (case["length"] + 1) * 0.5, case["nodes"])
        kept = nodes * degree * 0.1
        return {"bytes": nodes * degree * b + kept * (b + (8 if case["weights"] else 0)), "flops": 0}
    if kind == "dot":
        d = case["heads"] * case["dim"]
        rows = min(2.0 * case["edges"], 2.0 * case["nodes"])  # no more rows than there are nodes
        return {"bytes": rows * d * 4 + case["edges"] * (2 * b + 4 * case["heads"]),
                "flops": 2.0 * case["edges"] * d}
    if kind == "normalize":
        return {"bytes": case["edges"] * 8 + case["nodes"] * 12
                + (case["edges"] * 8 if case["axis"] else 0), "flops": 0}
    edges = case["edges"] + case["nodes"]
    return {"bytes": edges * (2 * b + b + 8) + case["nodes"] * 8, "flops": 0}


def tolerance(case):
    """Whole numbers are the same; sums and products of 32-bit floats may be added in another order."""
    if case["kind"] in ("ladies", "dot", "normalize"):
        return {"rel": 1e-5}
    return "exact"
