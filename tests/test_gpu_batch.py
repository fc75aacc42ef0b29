"""The batched form of a heterogeneous dataflow: its row-range ops against plain torch, and
whole models against the executor that runs one relation at a time."""
import pytest
import torch

import pipeline_cases as cases
from helpers import assert_close
from yitu_amd import _lib, graph_ext, xgnn_h
from yitu_amd.xgnn_h import ir, models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [1, 3, 4, 20, 64])
def test_fold_of_row_ranges(dev, width):
    g = torch.Generator().manual_seed(width)
    x = torch.randn(70, width, generator=g).to(dev).requires_grad_()
    # rows, sources, divisor, act, alpha: an empty range, one without sources, rows 45..49 unread
    ranges = [(5, [0, 30], 2.0, 0, 0.0), (0, [7], 1.0, 1, 0.0), (3, [], 1.0, 0, 0.0),
              (20, [50], 3.0, 1, 0.0), (10, [5, 15, 35], 1.0, 2, 0.7), (4, [25], 1.0, 2, 1.0)]
    plan = _lib.ops().fold_plan(70, ranges, x)
    out = _lib.ops().fold_rows(x, plan)
    want = []
    for rows, sources, div, act, alpha in ranges:
        v = sum((x[s:s + rows] for s in sources), torch.zeros(rows, width, device=dev)) / div
        want.append(v.relu() if act == 1 else torch.nn.functional.elu(v, alpha) if act == 2 else v)
    want = torch.cat(want)
    assert_close(out, want)
    dy = torch.randn(want.shape, generator=g).to(dev)
    assert_close(torch.autograd.grad(out, x, dy)[0], torch.autograd.grad(want, x, dy)[0])


@pytest.mark.parametrize("width,scale", [(64, 70_000), (3, 400_000), (256, 16_400), (7, 150_001)])
def test_fold_of_many_rows(dev, width, scale):
    """Sizes at which a thread takes several vectors: workgroups inside a range, across two and
    over a row of tiny ones, the last one not full, with every activation."""
    g = torch.Generator().manual_seed(width)
    rows = [scale, 3, 1, 5, scale // 3, 2, scale // 5 + 1]
    starts = torch.tensor([0] + [2 * r for r in rows]).cumsum(0).tolist()
    total = starts[-1] + 4
    ranges = [(r, [s, s + r][:1 + i % 2] + ([s + r] if i == 4 else []), (1.0, 3.0)[i % 2], i % 3, 0.8)
              for i, (r, s) in enumerate(zip(rows, starts))]
    x = torch.randn(total, width, generator=g).to(dev).requires_grad_()
    out = _lib.ops().fold_rows(x, _lib.ops().fold_plan(total, ranges, x))
    want = torch.cat([(lambda v: v.relu() if act == 1 else torch.nn.functional.elu(v, alpha)
                       if act == 2 else v)(sum(x[s:s + r] for s in sources) / div)
                      for r, sources, div, act, alpha in ranges])
    assert_close(out, want)
    dy = torch.randn(want.shape, generator=g).to(dev)
    assert_close(torch.autograd.grad(out, x, dy)[0], torch.autograd.grad(want, x, dy)[0])


@pytest.mark.parametrize("split", [False, True])
def test_fold_result_may_be_written_where_no_activation_made_it(dev, split):
    def run(ranges, write):
        x = torch.randn(12, 4, device=dev).requires_grad_()
        plan = _lib.ops().fold_plan(12, ranges, x)
        parts = _lib.ops().fold_split(x, plan, [5, 7]) if split else [_lib.ops().fold_rows(x, plan)]
        parts[write].mul_(3.0)
        return torch.autograd.grad([p.sum() for p in parts], x)[0]

    third = [(5, [0], 3.0, 0, 0.0), (7, [5], 3.0, 0, 0.0)]
    want = torch.full((12, 4), 1 / 3, device=dev)
    want[:5 if split else 12] = 1.0
    assert_close(run(third, 0), want)
    relu = [(5, [0], 1.0, 1, 0.0), (7, [5], 1.0, 0, 0.0)]
    with pytest.raises(RuntimeError, match="inplace"):
        run(relu, 0)
    if split:  # the part beside it is no result of the ReLU
        assert_close(run(relu, 1)[5:], torch.full((7, 4), 3.0, device=dev))


def test_fold_plan_refuses_ranges_outside_or_twice(dev):
    x = torch.zeros(10, 4, device=dev)
    with pytest.raises(RuntimeError):
        _lib.ops().fold_plan(10, [(4, [7], 1.0, 0, 0.0)], x)
    with pytest.raises(RuntimeError):
        _lib.ops().fold_plan(10, [(4, [0], 1.0, 0, 0.0), (4, [3], 1.0, 0, 0.0)], x)
    with pytest.raises(RuntimeError):
        _lib.ops().fold_rows(x, _lib.ops().fold_plan(9, [(9, [0], 1.0, 0, 0.0)], x))


@pytest.mark.parametrize("k,n", [(5, 3), (16, 32), (33, 17)])
@pytest.mark.parametrize("bias", [False, True])
def test_linear_over_row_ranges(dev, k, n, bias):
    """Rows read twice, not at all and in part, from two matrices."""
    g = torch.Generator().manual_seed(k)
    t = lambda *s: torch.randn(*s, generator=g).to(dev).requires_grad_()  # noqa: E731
    a, b = t(40, k), t(9, k)
    units = [(0, 0, 25), (1, 0, 9), (0, 20, 15), (0, 20, 1), (1, 0, 9)]
    ws, bs = [t(n, k) for _ in units], [t(n) for _ in units] if bias else []
    plan = _lib.ops().linear_plan(units, [bias] * len(units), [40, 9], a)
    y = _lib.ops().linear_rows([a, b], ws, bs, plan)
    want = torch.cat([(a, b)[m][o:o + r] @ w.t() + (bs[i] if bias else 0.0)
                      for i, ((m, o, r), w) in enumerate(zip(units, ws))])
    assert_close(y, want)
    dy = torch.randn(want.shape, generator=g).to(dev)
    leaves = [a, b, *ws, *bs]
    for got, ref in zip(torch.autograd.grad(y, leaves, dy), torch.autograd.grad(want, leaves, dy)):
        assert_close(got, ref, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("which", ["rgcn", "rgat"])
@pytest.mark.parametrize("stitch", [False, True])
@pytest.mark.parametrize("relations", [7, 3])  # several and single relations per type
def test_batched_model_equals_one_relation_at_a_time(dev, which, stitch, relations):
    torch.manual_seed(5)
    hgraph = cases.hetero_graph(device=dev)
    if relations == 3:
        kept = [("paper", "written_by", "author"), ("author", "writes", "paper"),
                ("paper", "appears_in", "venue")]
        hgraph = cases.mp.HeteroGraph.from_blocks(
            cases.NTYPES, {r: hgraph.hetero_graph[r].blk for r in kept}, device=dev)
    kwargs = cases.hetero_kwargs(hgraph, device=dev, with_norms=which == "rgcn")
    model = (models.RGCNModel(hgraph, 12, 16, 5) if which == "rgcn"
             else models.RGATModel(hgraph, 12, 16, 8, n_heads=2)).to(dev)
    flow = xgnn_h.Optimizer().lower(xgnn_h.Module2IR().transform(model, kwargs), kwargs)
    if stitch:
        flow = xgnn_h.Stitcher().transform(flow, kwargs)
    batched = xgnn_h.batch.batch_rows(flow, kwargs)
    ops = cases.ops_of(batched)
    core = "spmm" if which == "rgcn" else "gat"
    if stitch or relations == 3:
        assert ops[core + "_rows"] == 2 and ops[core] == 0 and ops["linear"] == 0
    params = list(model.parameters())
    weights = {}
    results = []
    for flag in (False, True):
        executor = xgnn_h.Executor(group_linears=flag)
        executor.eval()
        out = executor.run(flow, kwargs)
        for i, (k, v) in enumerate(out.items()):
            weights.setdefault(k, torch.randn_like(v))
        results.append((out, torch.autograd.grad([out[k] for k in out], params,
                                                 [weights[k] for k in out], allow_unused=True)))
        if flag:  # a second pass, and one with other parameters, on the same plans
            with torch.no_grad():
                for p in params:
                    p.mul_(1.1)
            again = executor.run(flow, kwargs)
            plain = xgnn_h.Executor(group_linears=False)
            plain.eval()
            for k, v in plain.run(flow, kwargs).items():
                assert_close(again[k], v, rtol=1e-4, atol=1e-5)
    (out_a, grads_a), (out_b, grads_b) = results
    for k in out_a:
        assert_close(out_b[k], out_a[k], rtol=1e-4, atol=1e-5)
    for a, b in zip(grads_a, grads_b):
        assert (a is None) == (b is None)
        if a is not None:
            assert_close(b, a, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("which", ["rgcn", "rgat"])
def test_forget_reaches_what_a_batched_model_keeps(dev, which):
    """Index and norm tensors refilled past torch's version counter and named to forget(): the
    executor's block-diagonal copies and edge weights are made again."""
    torch.manual_seed(2)
    hgraph = cases.hetero_graph(device=dev)
    kwargs = cases.hetero_kwargs(hgraph, device=dev, with_norms=which == "rgcn")
    model = (models.RGCNModel(hgraph, 12, 16, 5) if which == "rgcn"
             else models.RGATModel(hgraph, 12, 16, 8, n_heads=2)).to(dev)
    flow = xgnn_h.Optimizer().lower(xgnn_h.Module2IR().transform(model, kwargs), kwargs)
    executor, plain = xgnn_h.Executor(), xgnn_h.Executor(group_linears=False)
    for e in (executor, plain):
        e.eval()
    before = executor.run(flow, kwargs)
    for g in hgraph.hetero_graph.values():
        indices = g.blk.adj_sparse[1]
        version = indices._version
        indices.data.copy_((indices + 1) % g.blk.size[1])
        assert indices._version == version
        graph_ext.forget(*g.blk.adj_sparse)
    for norm in kwargs.get("norms", {}).values():
        norm.data.mul_(3.0)
        graph_ext.forget(norm)
    after, want = executor.run(flow, kwargs), plain.run(flow, kwargs)
    for t in want:
        assert_close(after[t], want[t], rtol=1e-4, atol=1e-5)
        assert not torch.allclose(after[t], before[t], rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("which", ["rgcn", "rgat"])
def test_outputs_of_a_batched_model_can_be_written_in_place(dev, which):
    torch.manual_seed(1)
    hgraph = cases.hetero_graph(device=dev)
    kwargs = cases.hetero_kwargs(hgraph, device=dev, with_norms=which == "rgcn")
    model = (models.RGCNModel(hgraph, 12, 16, 5) if which == "rgcn"
             else models.RGATModel(hgraph, 12, 16, 8, n_heads=2)).to(dev)
    flow = xgnn_h.Optimizer().lower(xgnn_h.Module2IR().transform(model, kwargs), kwargs)
    for form in (flow, xgnn_h.Stitcher().transform(flow, kwargs)):
        grads = []
        for flag in (False, True):
            executor = xgnn_h.Executor(group_linears=flag)
            executor.eval()
            out = executor.run(form, kwargs)
            out["paper"].mul_(2.0)
            out["venue"].add_(1.0)
            grads.append(torch.autograd.grad([v.square().sum() for v in out.values()],
                                             list(model.parameters()), allow_unused=True))
        for a, b in zip(*grads):
            assert (a is None) == (b is None)
            if a is not None:
                assert_close(b, a, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("which", ["rgcn", "rgat"])
@pytest.mark.parametrize("stitch", [False, True])
def test_batched_model_in_training_mode(dev, which, stitch, monkeypatch):
    """Dropout between the layers: with a mask that depends on the values alone the batched form
    gives the outputs and gradients of one relation at a time, stitched or not."""
    torch.manual_seed(3)
    hgraph = cases.hetero_graph(device=dev)
    kwargs = cases.hetero_kwargs(hgraph, device=dev, with_norms=which == "rgcn")
    model = (models.RGCNModel(hgraph, 12, 16, 5) if which == "rgcn"
             else models.RGATModel(hgraph, 12, 16, 8, n_heads=2)).to(dev)
    flow = xgnn_h.Optimizer().lower(xgnn_h.Module2IR().transform(model, kwargs), kwargs)
    if stitch:
        flow = xgnn_h.Stitcher().transform(flow, kwargs)
    batched = xgnn_h.batch.batch_rows(flow, kwargs, training=True)
    assert cases.ops_of(batched)["dropout"] == 1  # one draw for all node types
    drawn = []

    def dropout(x, p, training):
        assert p == 0.5 and training
        drawn.append(x.size(0))
        return x * (x > -0.05) / (1 - p)

    monkeypatch.setattr(torch.nn.functional, "dropout", dropout)
    results, weights = [], {}
    for flag in (False, True):
        executor = xgnn_h.Executor(group_linears=flag)
        executor.train()
        del drawn[:]
        out = executor.run(flow, kwargs)
        assert sum(drawn) == sum(cases.NTYPES.values()) and len(drawn) == (1 if flag else 3)
        for k, v in out.items():
            weights.setdefault(k, torch.randn_like(v))
        results.append([out[k] for k in weights] + list(torch.autograd.grad(
            [out[k] for k in weights], list(model.parameters()), list(weights.values()),
            allow_unused=True)))
    for a, b in zip(*results):
        assert (a is None) == (b is None)
        if a is not None:
            assert_close(b, a, rtol=1e-4, atol=1e-4)


def test_two_dropouts_of_the_same_rows_differ(dev):
    """F.dropout(h, .5) - F.dropout(h, .5): about half of the entries
    are not zero, whatever the batch."""
    hgraph = cases.hetero_graph(device=dev)
    kwargs = cases.hetero_kwargs(hgraph, device=dev)

    class Model(models.RGCNModel):
        def forward(self, hgraph, norms, xs):
            drop = lambda h: torch.nn.functional.dropout(h, 0.5)  # noqa: E731
            return {t: drop(h) - drop(h) for t, h in self._run(hgraph, xs, norms).items()}

    model = Model(hgraph, 8, 8, 16).to(dev)
    flow = xgnn_h.Optimizer().lower(xgnn_h.Module2IR().transform(model, kwargs), kwargs)
    executor = xgnn_h.Executor()
    executor.train()
    for form in (flow, xgnn_h.Stitcher().transform(flow, kwargs)):
        out = executor.run(form, kwargs)
        share = torch.cat(list(out.values())).ne(0).float().mean()
        assert 0.4 < float(share) < 0.6  # 117 x 16 fair draws: a standard error of 0.012


def test_batched_model_in_training_mode_keeps_its_shapes(dev):
    hgraph = cases.hetero_graph(device=dev)
    kwargs = cases.hetero_kwargs(hgraph, device=dev)
    model = models.RGCNModel(hgraph, 8, 8, 4).to(dev)
    flow = xgnn_h.Module2IR().transform(model, kwargs)
    executor = xgnn_h.Executor()
    executor.train()  # dropout is drawn for the whole batch
    out = executor.run(flow, kwargs)
    assert {k: list(v.shape) for k, v in out.items()} == \
        {k: [n, 4] for k, n in hgraph.nty2num.items()}
    assert isinstance(flow, dict) and all(isinstance(n, ir.Node) for n in flow.values())
