"""The work that users of this package have it do, stated as timed cases.

Every case goes through the public entry points: the conv modules over the module-1
ops, the attention layers, the op pairs of ``graph_ext``, the heterogeneous layers in
both precisions, a captured and stitched heterogeneous model, temporal sampling with its
attention layer, and the preparation of a graph from its edge list. Training passes
return the outputs and every gradient. Node counts, degrees and widths span what the
configurations, tests and benchmark of this repository use, ragged ones included; ids of
the skewed graphs are relabelled at random, as real vertex ids carry no structure.
"""
import math
import types

import numpy as np
import torch

from yitu_amd import YiTu_GNN_kernel, graph_ext, sampler_core, xgnn_h
from yitu_amd.data import csr, graphgen
from yitu_amd.nn import GCNConv, GINConv
from yitu_amd.temporal import TemporalBlock, TransfomerAttentionLayer, build_tcsr
from yitu_amd.utils.input_info import InputInfo
from yitu_amd.xgnn_h import block as xblock
from yitu_amd.xgnn_h import layers as xlayers
from yitu_amd.xgnn_h import models, mp

DEV = "cuda"
PART_SIZE = 32


def listed():
    return [
        # a citation-scale graph: wide input features to a narrow hidden layer, launch-bound
        dict(name="gcn_small", kind="gcn", graph="uniform", nodes=3000, degree=4, d_in=500, d_out=16),
        # a mid-size graph with communities (what a vertex reorder leaves), odd layer widths
        dict(name="gin_ragged", kind="gin", graph="communities", nodes=150_000, degree=15, d_in=100,
             d_out=47),
        # the large power-law graph of the benchmark, 128 features
        dict(name="gcn_large", kind="gcn", graph="skewed", nodes=1 << 21, degree=30, d_in=128,
             d_out=128),
        # the usual first attention layer on a citation-scale graph: 8 heads of 8
        dict(name="gat_small", kind="gat", graph="uniform", nodes=3000, degree=4, d_in=500, heads=8,
             width=8),
        # a mid-size graph, 128 hidden floats in 4 heads
        dict(name="gat_mid", kind="gat", graph="communities", nodes=100_000, degree=20, d_in=100,
             heads=4, width=32),
        # the attention configuration of the benchmark: 2^18 nodes, 13 M draws, 4 heads of 64
        dict(name="gat_large", kind="gat", graph="skewed", nodes=1 << 18, degree=50, d_in=256,
             heads=4, width=64),
        # attention spelled with the two separate ops and their backwards, odd head shape
        dict(name="attention_ops", kind="attention_ops", graph="skewed", nodes=50_000, degree=18,
             heads=3, width=20),
        # a relational layer, fp32: per-type products and one stacked aggregation
        dict(name="rgcn_f32", kind="rgcn", dtype="f32", nodes=120_000, types=4, relations=8, degree=8,
             d_in=192, d_out=96),
        # the relational configuration of the benchmark in bf16
        dict(name="rgcn_bf16", kind="rgcn", dtype="bf16", nodes=491_520, types=4, relations=8,
             degree=8, d_in=256, d_out=256),
        # a whole two-layer relational model, captured, lowered and stitched: many small launches
        dict(name="hetero_model", kind="hetero_model", model="rgcn", nodes=7262, types=5, relations=10,
             edges=48_810, hidden=32),
        # one batch of temporal attention: sampling on the device, gather, layer, gradients
        dict(name="temporal", kind="temporal", nodes=1 << 17, events=1 << 20, batch=2048, fan=20,
             d_node=172, d_edge=0, d_time=100, heads=1, d_out=100),
        # a new graph: edge list to CSR, edge scales, by-source view and row plans
        dict(name="graph_prep", kind="graph_prep", graph="skewed", nodes=200_000, degree=15),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _graph(rng, most_nodes, most_edges, least_nodes=1000):
    nodes = _log(rng, least_nodes, most_nodes)
    degree = _log(rng, 3, max(3, min(50, most_edges // nodes)))
    return dict(graph=rng.choice(["uniform", "skewed", "communities"]), nodes=nodes, degree=degree)


def draw(rng):
    kind = rng.choice(["gcn", "gin", "gat", "gat", "attention_ops", "rgcn", "rgcn", "hetero_model",
                       "temporal", "graph_prep"])
    if kind in ("gcn", "gin"):
        d_in, d_out = _log(rng, 16, 512), _log(rng, 7, 256)
        most = min(1 << 20, (1 << 35) // (d_in * d_out), (1 << 29) // (d_in + d_out))
        return dict(kind=kind, **_graph(rng, most, 20_000_000), d_in=d_in, d_out=d_out)
    if kind == "gat":
        heads, width = rng.choice([(1, 16), (1, 40), (1, 128), (2, 24), (2, 64), (4, 8), (4, 32), (4, 64),
                                   (8, 8), (8, 16), (8, 32)])
        return dict(kind=kind, **_graph(rng, 1 << 18, 5_000_000), d_in=_log(rng, 16, 512), heads=heads,
                    width=width)
    if kind == "attention_ops":
        return dict(kind=kind, **_graph(rng, 1 << 18, 5_000_000), heads=rng.choice([1, 2, 3, 4, 5, 8]),
                    width=_log(rng, 5, 64))
    if kind == "rgcn":
        types_ = rng.randint(2, 5)
        out = dict(kind=kind, dtype=rng.choice(["f32", "bf16"]), nodes=_log(rng, 5000, 400_000),
                   types=types_, relations=types_ + rng.randint(0, 5), degree=rng.randint(2, 12))
        widths = [32, 64, 96, 128, 136, 192, 256]
        return dict(out, d_in=rng.choice(widths), d_out=rng.choice(widths))
    if kind == "hetero_model":
        model = rng.choice(["rgcn", "rgat"])  # an attention relation has three Linears
        types_ = rng.randint(2, 6 if model == "rgcn" else 3)
        relations = types_ + rng.randint(0, 4 if model == "rgcn" else 1)
        return dict(kind=kind, model=model, nodes=_log(rng, 2000, 40_000), types=types_, relations=relations,
                    edges=_log(rng, 10_000, 200_000), hidden=rng.choice([16, 32, 64]))
    if kind == "temporal":
        heads, d_out = rng.choice([(1, 100), (2, 100), (1, 64), (2, 128), (4, 172)])
        return dict(kind=kind, nodes=_log(rng, 5000, 1 << 17), events=_log(rng, 50_000, 1 << 20),
                    batch=2 * _log(rng, 50, 2000), fan=rng.randint(5, 25),
                    d_node=rng.choice([100, 128, 172]), d_edge=rng.choice([0, 0, 50, 172]),
                    d_time=rng.choice([64, 100]), heads=heads, d_out=d_out)
    return dict(kind=kind, **_graph(rng, 1 << 20, 16_000_000))


# ---- inputs ---------------------------------------------------------------------------


def _edges(c, seed, gen):
    """nodes * degree distinct (src, dst) pairs of the case's graph, self loops among them,
    sorted by destination: the count is the same for every seed."""
    n, m = c["nodes"], c["nodes"] * c["degree"]
    if c["graph"] == "uniform":
        src, dst = graphgen.erdos_renyi(n, m, seed, self_loops=False, device=DEV)
    elif c["graph"] == "communities":
        size = 512 if n >= 8192 else 64
        inside = max(1, c["degree"] // 2)
        src, dst = graphgen.planted_partition(-(-n // size), size, inside, max(1, c["degree"] - inside),
                                              seed, device=DEV)
        keep = (src < n) & (dst < n)
        src, dst = src[keep], dst[keep]
    else:
        scale = max(1, (n - 1).bit_length())
        src, dst = graphgen.rmat(scale, m, seed, device=DEV)
        perm = torch.randperm(1 << scale, generator=gen, device=DEV) % n
        src, dst = perm[src], perm[dst]
    loops = torch.arange(n, device=DEV) * (n + 1)
    keys = torch.unique(torch.cat([dst * n + src, loops]))
    while keys.numel() < m:  # what merging took away
        more = torch.randint(0, n * n, (m - keys.numel() + 64,), generator=gen, device=DEV)
        keys = torch.unique(torch.cat([keys, more]))
    surplus = torch.randperm(keys.numel(), generator=gen, device=DEV)[:keys.numel() - m]
    keep = torch.ones(keys.numel(), dtype=torch.bool, device=DEV)
    keep[surplus] = False
    keys = keys[keep]
    dst = torch.div(keys, n, rounding_mode="floor")
    return keys - dst * n, dst


def _csr(c, seed, gen):
    src, dst = _edges(c, seed, gen)
    indptr = torch.zeros(c["nodes"] + 1, dtype=torch.int64, device=DEV)
    indptr[1:] = torch.cumsum(torch.bincount(dst, minlength=c["nodes"]), 0)
    return indptr.to(torch.int32), src.to(torch.int32)


def _normal(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEV)


def _conv_state(c, seed, gen):
    indptr, indices = _csr(c, seed, gen)
    dataset = types.SimpleNamespace(num_nodes=c["nodes"], avg_degree=c["degree"], avg_edgeSpan=0.0,
                                    num_features=c["d_in"])
    info = InputInfo(indptr, indices, graphgen.gcn_norm(indptr), PART_SIZE, 32, 8, 100, c["d_out"], dataset)
    info.partPtr, info.part2Node = YiTu_GNN_kernel.build_part(PART_SIZE, indptr)
    conv = (GCNConv if c["kind"] == "gcn" else GINConv)(c["d_in"], c["d_out"]).to(DEV)
    if c["kind"] == "gcn":
        info.prepare_edge_scale()
    x = _normal(gen, c["nodes"], c["d_in"]).requires_grad_()
    return dict(conv=conv, info=info, x=x, grad=_normal(gen, c["nodes"], c["d_out"]))


def _gat_state(c, seed, gen):
    indptr, indices = _csr(c, seed, gen)
    layer = xlayers.GATLayer(c["d_in"], c["width"], c["heads"]).to(DEV)
    x = _normal(gen, c["nodes"], c["d_in"]).requires_grad_()
    return dict(layer=layer, blk=xblock.Block([c["nodes"], c["nodes"]], [indptr, indices]), x=x,
                grad=_normal(gen, c["nodes"], c["width"]))


def _attention_ops_state(c, seed, gen):
    indptr, indices = _csr(c, seed, gen)
    n, h, f = c["nodes"], c["heads"], c["width"]
    return dict(indptr=indptr, indices=indices, query=_normal(gen, 1, n, h), key=_normal(gen, n, h),
                x=_normal(gen, n, h, f), grad=_normal(gen, n, h, f))


def _type_sizes(c):
    # halving from type to type, as in the relational configuration
    share = [0.5 ** t for t in range(c["types"])]
    return [max(8, int(c["nodes"] * s / sum(share))) for s in share]


def _relations(c, seed, degree):
    """{(source type, relation, destination type): Block}: every type is reached."""
    sizes = _type_sizes(c)
    blocks = {}
    for r in range(c["relations"]):
        d_t, s_t = r % c["types"], (r + 1 + r // c["types"]) % c["types"]
        indptr, indices = graphgen.bipartite_uniform(sizes[d_t], sizes[s_t], degree(sizes[d_t]), seed + r,
                                                     device=DEV)
        blk = xblock.Block([sizes[d_t], sizes[s_t]], [indptr, indices])
        blk.right_norm = xlayers.right_norm(blk)
        blocks[("t%d" % s_t, "r%d" % r, "t%d" % d_t)] = blk
    return sizes, blocks


def _rgcn_state(c, seed, gen):
    sizes, blocks = _relations(c, seed, lambda n_dst: c["degree"])
    ntypes = {"t%d" % t: n for t, n in enumerate(sizes)}
    layer = xlayers.StackedHeteroGCN(ntypes, list(blocks), c["d_in"], c["d_out"], per_relation=False).to(DEV)
    stacked = layer.stack(blocks, {str(k): b.right_norm for k, b in blocks.items()})
    xs = {t: _normal(gen, n, c["d_in"]) for t, n in ntypes.items()}
    grads = _normal(gen, sum(sizes), c["d_out"])
    if c["dtype"] == "f32":
        return dict(layer=layer, xs={t: x.requires_grad_() for t, x in xs.items()},
                    grads=dict(zip(ntypes, grads.split(sizes))))
    weights = [layer.fcs[t].weight.detach().to(torch.bfloat16).contiguous() for t in ntypes]
    return dict(stacked=stacked, sizes=sizes, weights=weights, xs=[x.to(torch.bfloat16) for x in xs.values()],
                grads=grads.to(torch.bfloat16), d_out=c["d_out"])


def _hetero_model_state(c, seed, gen):
    sizes, blocks = _relations(c, seed, lambda n_dst: c["edges"] / c["relations"] / n_dst)
    ntypes = {"t%d" % t: n for t, n in enumerate(sizes)}
    hgraph = mp.HeteroGraph.from_blocks(ntypes, blocks, device=DEV)
    kwargs = {"hgraph": hgraph, "xs": {t: torch.arange(n, device=DEV) for t, n in ntypes.items()}}
    d = c["hidden"]
    if c["model"] == "rgcn":
        model = models.RGCNModel(hgraph, d, d, d).to(DEV)
        kwargs["norms"] = {str(rel): g.right_norm() for rel, g in hgraph.hetero_graph.items()}
    else:
        model = models.RGATModel(hgraph, d, d, d, n_heads=2).to(DEV)
    flow = xgnn_h.Optimizer().lower(xgnn_h.Module2IR().transform(model, kwargs), kwargs)
    flow = xgnn_h.Stitcher().transform(flow, kwargs)
    executor = xgnn_h.Executor()
    executor.eval()
    return dict(executor=executor, flow=flow, kwargs=kwargs, params=list(model.parameters()),
                grads={t: _normal(gen, n, d) for t, n in ntypes.items()})


def _temporal_state(c, seed, gen):
    rng = np.random.default_rng(seed)
    n, m = c["nodes"], c["events"]
    src, dst = ((rng.zipf(1.2, m) - 1) % n for _ in range(2))
    when = np.sort(rng.uniform(0, 1e6, m)).astype(np.float32)
    tcsr = build_tcsr(*(torch.as_tensor(a).to(DEV) for a in (src, dst, when)), n)
    sampler = sampler_core.GpuParallelSampler(*(t.cpu().numpy() for t in tcsr), 16, 1, 1, [c["fan"]], True,
                                              False, 1, 0.0, device=DEV)
    picked = rng.integers(m * 9 // 10, m, c["batch"] // 2)
    layer = TransfomerAttentionLayer(c["d_node"], c["d_edge"], c["d_time"], c["heads"], 0.0, 0.0,
                                     c["d_out"]).to(DEV)
    roots = torch.as_tensor(np.concatenate([src[picked], dst[picked]]), dtype=torch.int32)
    return dict(sampler=sampler, layer=layer, memory=_normal(gen, n, c["d_node"]),
                edge_feat=_normal(gen, m, c["d_edge"]) if c["d_edge"] else None, roots=roots.to(DEV),
                root_ts=torch.as_tensor(np.concatenate([when[picked], when[picked]])).to(DEV),
                grad=_normal(gen, 2 * len(picked), c["d_out"]))


def _graph_prep_state(c, seed, gen):
    src, dst = _edges(c, seed, gen)
    # an edge list as it is read: any order, an eighth of the edges twice
    order = torch.randperm(src.numel() * 9 // 8, generator=gen, device=DEV) % src.numel()
    return dict(nodes=c["nodes"], src=src[order], dst=dst[order])


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    torch.manual_seed(seed)  # the layers' own initialisation
    make = {"gcn": _conv_state, "gin": _conv_state, "gat": _gat_state, "attention_ops": _attention_ops_state,
            "rgcn": _rgcn_state, "hetero_model": _hetero_model_state, "temporal": _temporal_state,
            "graph_prep": _graph_prep_state}[case["kind"]]
    return dict(make(case, seed, gen), kind=case["kind"], dtype=case.get("dtype", "f32"))


# ---- one pass -------------------------------------------------------------------------


def _run_rgcn_bf16(s):
    (blk, values), d = s["stacked"], s["d_out"]
    indptr, indices = blk.adj_sparse
    n = sum(s["sizes"])
    h = torch.empty(n, d, dtype=torch.bfloat16, device=DEV)
    graph_ext.gemm_bf16_typed(s["xs"], s["weights"], trans_b=True, out_list=list(h.split(s["sizes"])))
    out = graph_ext.spmm_forward(values, indptr, indices, h.view(n, 1, d), out_dtype=torch.bfloat16)
    dh = graph_ext.spmm_backward(values, indptr, indices, h.view(n, 1, d), s["grads"].view(n, 1, d),
                                 need_grad_a=False, grad_x_dtype=torch.bfloat16)[1]
    parts = list(dh.view(n, d).split(s["sizes"]))
    dws = graph_ext.gemm_bf16_tn_typed(parts, s["xs"])
    dxs = graph_ext.gemm_bf16_typed(parts, s["weights"], out_dtype=torch.bfloat16)
    return [out, *dws, *dxs]


def _run_attention_ops(s):
    indptr, indices, query, key, x = s["indptr"], s["indices"], s["query"], s["key"], s["x"]
    attn = graph_ext.sddmm_forward(indptr, indices, query, key)
    out = graph_ext.spmm_forward(attn, indptr, indices, x)
    grad_attn, grad_x = graph_ext.spmm_backward(attn, indptr, indices, x, s["grad"])
    grad_query, grad_key = graph_ext.sddmm_backward(indptr, indices, query, key, attn, grad_attn)
    return [attn, out, grad_x, grad_query, grad_key]


def _run_temporal(s):
    s["sampler"].sample(s["roots"], s["root_ts"])
    sampled = s["sampler"].get_ret()[0]
    blk = TemporalBlock.from_device_block(sampled, s["memory"])
    if s["edge_feat"] is not None:
        blk.f = s["edge_feat"][sampled.eid().to(torch.int64)]
    out = s["layer"](blk)  # node features are inputs: the gradients are the parameters'
    return [out, *torch.autograd.grad(out, list(s["layer"].parameters()), s["grad"])]


def _run_graph_prep(s):
    indptr, indices = csr.coo_to_csr(s["dst"], s["src"], s["nodes"])
    scale = YiTu_GNN_kernel.edge_scale(indices, graphgen.gcn_norm(indptr))
    t = graph_ext.transposed(indptr, indices, s["nodes"])
    return [indptr, indices, scale, t.t_indptr, t.t_rows, t.t_perm]


def run(s):
    kind = s["kind"]
    if kind in ("gcn", "gin"):
        out = s["conv"](s["x"], s["info"])
        return [out, *torch.autograd.grad(out, [s["x"], s["conv"].weights], s["grad"])]
    if kind == "gat":
        out = s["layer"](s["blk"], s["x"])
        return [out, *torch.autograd.grad(out, [s["x"], *s["layer"].parameters()], s["grad"])]
    if kind == "attention_ops":
        return _run_attention_ops(s)
    if kind == "rgcn" and s["dtype"] == "bf16":
        return _run_rgcn_bf16(s)
    if kind == "rgcn":
        outs = s["layer"](s["xs"])
        names = list(outs)
        grads = torch.autograd.grad([outs[t] for t in names], [*s["xs"].values(), *s["layer"].parameters()],
                                    [s["grads"][t] for t in names])
        return [*(outs[t] for t in names), *grads]
    if kind == "hetero_model":
        outs = s["executor"].run(s["flow"], s["kwargs"])
        names = list(outs)
        grads = torch.autograd.grad([outs[t] for t in names], s["params"], [s["grads"][t] for t in names],
                                    allow_unused=True)
        return [*(outs[t] for t in names), *grads]
    if kind == "temporal":
        return _run_temporal(s)
    return _run_graph_prep(s)


# ---- what a pass cannot do without ----------------------------------------------------


def work(case):
    """Inputs read once and outputs written once, forward and backward; products and
    per-edge multiply-adds."""
    c, kind = case, case["kind"]
    n = c["nodes"]
    if kind in ("gcn", "gin"):
        e, a, b = n * c["degree"], c["d_in"], c["d_out"]
        gathered = b if kind == "gcn" else a  # GCN aggregates X.W, GIN aggregates X
        return {"bytes": 4 * (2 * n + e) + 4 * n * (2 * a + 2 * b) + 8 * a * b,
                "flops": 6 * n * a * b + 4 * e * gathered}
    if kind == "gat":
        e, a, h, w = n * c["degree"], c["d_in"], c["heads"], c["heads"] * c["width"]
        return {"bytes": 4 * (n + 2 * e) + 4 * n * (2 * a + 2 * c["width"]) + 8 * a * w,
                "flops": 6 * n * a * w + 6 * n * w * 2 * h + 6 * e * w + 30 * e * h}
    if kind == "attention_ops":
        e, h, w = n * c["degree"], c["heads"], c["heads"] * c["width"]
        return {"bytes": 4 * (n + 3 * e) + 4 * e * h + 4 * n * (4 * w + 4 * h), "flops": 6 * e * w + 30 * e * h}
    if kind == "rgcn":
        sizes = _type_sizes(c)
        e = sum(sizes[r % c["types"]] * c["degree"] for r in range(c["relations"]))
        n, a, b, size = sum(sizes), c["d_in"], c["d_out"], 2 if c["dtype"] == "bf16" else 4
        return {"bytes": size * n * (2 * a + 2 * b) + (size + 4) * c["types"] * a * b + 4 * (n + 3 * e),
                "flops": 6 * n * a * b + 4 * e * b}
    if kind == "hetero_model":
        e, d = c["edges"], c["hidden"]
        wide = d if c["model"] == "rgcn" else 2 * d
        rows = c["relations"] * n / c["types"]  # rows that a layer's relations transform
        return {"bytes": 4 * (3 * n * d + 4 * c["relations"] * d * wide + 3 * e),
                "flops": 2 * 6 * rows * d * wide + 2 * 4 * e * wide}
    if kind == "temporal":
        b, k, dn, de, dt, o = c["batch"], c["fan"], c["d_node"], c["d_edge"], c["d_time"], c["d_out"]
        e = b * k
        return {"bytes": 4 * ((b + e) * dn + e * (de + 6) + 2 * b * o + 4 * o * (dn + de + dt)),
                "flops": 6 * (e * 2 * (dn + de + dt) + b * (2 * dn + dt + o)) * o + 12 * e * o}
    e = n * c["degree"]
    return {"bytes": 16 * (e * 9 // 8) + 4 * (4 * e + 3 * n), "flops": 0}


def tolerance(case):
    if case["kind"] == "graph_prep":
        return "exact"
    if case.get("dtype") == "bf16":
        return {"rel": 1e-2}
    return {"rel": 1e-5}
