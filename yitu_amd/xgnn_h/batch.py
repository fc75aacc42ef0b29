"""Batched form of a heterogeneous dataflow. A relational model applies one small product
and one small aggregation per relation (YiTu_GNN/YiTu_H/test/common/model.py:137-171): at the
scale of the reference's benchmark hundreds of launches of a few microseconds, issued more
slowly than the GPU runs them. Here the nodes of a dataflow that do the same thing and do
not depend on each other run together, each group as one launch:

* ``typed_rows``: Linears of one weight shape, all results in one buffer, one below the other;
* ``spmm_rows`` / ``gat_rows``: aggregations / attentions over one block-diagonal CSR whose
  columns point straight into the buffer that the members' features already share (nothing is
  concatenated), one row per destination, for attention one per (relation, destination);
* ``fold``: what follows up to the next product: the sum over a type's relations, the
  division by their number, ReLU / ELU.

A value is described by the rows of a batched result that hold it (``_Value``), so views,
squeezes, concatenations and selections cost nothing; only a reader outside the batched kinds
gets its rows as a tensor of their own. Groups form as dynamic batching does it: whatever can
be answered without a launch is, then the class with the shallowest ready nodes runs all of
them."""
import math

import torch
from torch.nn import functional as F

from . import block, ir, mp
from .stitcher import _is_add, _match_term

MAX_COLUMNS = 1 << 24  # what a packed CSR holds (block.py:53)
# Attention models whose products have this many rows on average run one relation at a time: the
# launches that a batch saves no longer count, while its few-column query and key products go
# through the grouped GEMM instead of the kernel that reads x once, and the by-source pass writes the
# rows of all destinations too. Forward and backward, ms, batched against one at a time: 256 -> 4 x 64
# with 200,000 rows a product 9.1 : 8.2, 123,000 21.2 : 21.0 (stitched 21.2 : 22.2), 60,000
# 13.1 : 14.8; 128 -> 4 x 32 with 333,000 14.3 : 13.1. (Without attention the batch is the faster one
# at every size: 256 wide, 491,520 nodes 13.8 : 16.3, stitched 13.4 : 13.3; 400,000 6.3 : 6.6.)
MANY_ROWS = 1 << 17

_FOLD_ACT = {"relu": 1, "elu": 2}
_ROWWISE = ("relu", "elu", "leaky_relu", "tanh", "sigmoid", "gelu", "div", "mul", "multiply")
# A slice of a batch (``rows``) read by an op that is no part of it gets its gradient through a
# zero-filled buffer of the batch's full height: a node's launches and 0.64 us per MB of the batch
# (16 slices of 1 GB made a step of 14.3 ms 24.6), against a node's launches and host work, about
# 20 us in both directions, for each that the batch does without.
CUT_US_PER_BYTE, US_PER_NODE = 6.4e-7, 20.0


class _Value:
    """Where the result of a node of the original dataflow is: rows ``segs`` (offset, rows), in
    order, of ``node``; or all of ``node`` (``segs`` None). ``blocks`` > 0: the parts of a
    ``stack``, one segment each."""
    __slots__ = ("node", "segs", "blocks")

    def __init__(self, node, segs=None, blocks=0):
        self.node, self.segs, self.blocks = node, segs, blocks


def _merge(segs):
    """Neighbouring segments joined."""
    out = []
    for off, n in segs:
        if out and out[-1][0] + out[-1][1] == off:
            out[-1] = (out[-1][0], out[-1][1] + n)
        elif n:
            out.append((off, n))
    return out


def _scalar_call(node):
    """The number of a ``fn(x, number)`` call, else None."""
    args = node.attrs["args"]
    if len(args) == 2 and isinstance(args[0], ir.Slot) and isinstance(args[1], (int, float)) and \
            not node.attrs["kwargs"]:
        return float(args[1])
    return None


def weights_of(node):
    """[(weight, bias)] of a product node."""
    a = node.attrs
    if node.op == "linear":
        return [(a["weight"], a["bias"])]
    return list(zip(a["weights"], a["biases"]))


class _Batcher:
    def __init__(self, dataflow, kwargs, training):
        self.training = training
        self.flow = self._scales_to_edges(dataflow, kwargs)
        self.order = ir.walk(self.flow)
        self.roots = ir.roots_of(self.flow)
        self.readers = {}
        for n in self.order:
            for c in {id(c): c for c in n.inputs.values()}.values():
                self.readers.setdefault(id(c), []).append(n)
        self.is_root = {id(r) for r in self.roots}
        self.value, self.parts, self.memo = {}, {}, {}
        self.together = False  # a group of two or more has been joined
        self.attention, self.unit_rows = False, []  # of the joined groups
        self.depth = {}
        for n in self.order:
            self.depth[id(n)] = 1 + max([self.depth[id(c)] for c in n.inputs.values()], default=0)
        self.query_side = self._query_side()

    # -- preparation ------------------------------------------------------------------
    @staticmethod
    def _scales_to_edges(dataflow, kwargs):
        """``norm * squeeze(spmm(g, x))`` of a relation on its own (model.py:30) becomes an
        aggregation with the scale as edge weight, the form that stitched relations have."""
        uses = ir.use_counts(dataflow)
        single = set()

        def rule(node, original):
            if uses.get(id(original), 0) == 1:
                single.add(id(node))
            term = _match_term(node, kwargs) if node.op == "call" else None
            if term is None or term.scale is None or term.core.op != "spmm" or \
                    "e" in term.core.inputs or term.post is None or \
                    term.post.fn_name() != "squeeze" or id(term.core) not in single or \
                    id(term.post) not in single or term.core.inputs["x"].size[1] != 1:
                return node
            g = term.core.inputs["g"]
            n_edges = kwargs[term.hgraph_key].hetero_graph[
                tuple(kwargs[term.hgraph_key].idx2rel[term.rel_index])].num_edges()
            weights = ir.Node("edge_values", {"g": g, "0": term.scale}, size=[n_edges, 1])
            core = ir.Node("spmm", {"g": g, "x": term.core.inputs["x"], "e": weights},
                           size=term.core.size)
            (slot,) = term.post.inputs
            return term.post.with_inputs({slot: core})

        return ir.rewrite(dataflow, rule)

    def _query_side(self):
        """Nodes on the way to an attention's query: they go first in their group, so that all
        queries of a batched attention end up in one row range."""
        marked = set()
        for n in reversed(self.order):
            if n.op in ("gat", "sddmm"):
                marked.add(id(n.inputs["q"]))
            if id(n) in marked and n.op in ("select", "stack", "concat", "linear", "bundle", "call"):
                marked.update(id(c) for c in n.inputs.values())
        return marked

    # -- values ------------------------------------------------------------------------
    @staticmethod
    def _rows_of(node):
        return int(node.size[0])

    def _segs(self, v):
        return v.segs if v.segs is not None else [(0, self._rows_of(v.node))]

    def _tensor(self, original):
        """The node whose result is ``original``'s, whole."""
        v = self.value[id(original)]
        if v.segs is None:
            return v.node
        segs = v.segs if v.blocks else _merge(v.segs)
        if not v.blocks and segs == [(0, self._rows_of(v.node))]:
            return v.node
        key = (id(v.node), tuple(segs), v.blocks)
        if key not in self.memo:
            tail = v.node.size[1:]
            pieces = [ir.Node("rows", {"x": v.node}, {"first": o, "rows": n}, [n] + tail)
                      for o, n in segs]
            if v.blocks:
                made = ir.Node("stack", {str(i): p for i, p in enumerate(pieces)},
                               size=[len(pieces)] + pieces[0].size)
            elif len(pieces) == 1:
                made = pieces[0]
            else:
                made = ir.Node("concat", {str(i): p for i, p in enumerate(pieces)},
                               size=[sum(n for _, n in segs)] + tail)
            self.memo[key] = made
        return self.memo[key]

    def _whole_batch(self, node, v, tail):
        """``node`` (a per-row function of one value) applied to all rows of the batch the value
        lives in, once."""
        (slot,), attrs = node.inputs, node.attrs
        if node.op == "call":
            slot = attrs["args"][0].key
            if node.fn_name() in ("view", "reshape", "squeeze"):
                slot, attrs = "0", {"fn": torch.Tensor.view, "kwargs": {},
                                    "args": (ir.Slot("0"), [-1] + list(tail))}
        key = (id(v.node), node.op, str(attrs))
        if node.op == "dropout":
            # each dropout draws for itself: one draw over the batch serves dropouts of
            # different rows, never two of the same row
            draws = self.memo.setdefault(key, [])
            made = next((d for d in draws if not any(self._overlap(s, v.segs) for s in d[1])), None)
            if made is None:
                made = (ir.Node("dropout", {slot: v.node}, attrs, [self._rows_of(v.node)] + list(tail)), [])
                draws.append(made)
            made[1].append(v.segs)
            return _Value(made[0], v.segs)
        if key not in self.memo:
            self.memo[key] = ir.Node(node.op, {slot: v.node}, attrs,
                                     [self._rows_of(v.node)] + list(tail))
        return _Value(self.memo[key], v.segs)

    @staticmethod
    def _overlap(a, b):
        return any(x < y + m and y < x + n for x, n in a for y, m in b)

    # -- nodes that need no batch ----------------------------------------------------------
    def _immediate(self, node):
        op = node.op
        if op in ("input", "graph"):
            return _Value(node)
        if op == "select" and id(node.inputs["x"]) in self.parts:
            return self.parts[id(node.inputs["x"])][node.attrs["index"]]
        if op in ("concat", "stack"):
            vs = [self.value[id(node.inputs[str(i)])] for i in range(len(node.inputs))]
            if all(v.segs is not None and v.node is vs[0].node and not v.blocks for v in vs) and \
                    all(len(v.segs) == 1 or op == "concat" for v in vs):
                return _Value(vs[0].node, [s for v in vs for s in v.segs],
                              len(vs) if op == "stack" else 0)
        if len(node.inputs) == 1 and op in ("call", "dropout"):
            (child,) = node.inputs.values()
            v = self.value[id(child)]
            if op == "dropout" and (not self.training or node.attrs["p"] == 0):
                return v
            if v.segs is not None and not v.blocks and node.size is not None and \
                    node.size[0] == child.size[0]:
                fn = node.fn_name() if op == "call" else "dropout"
                if fn in ("view", "reshape") and self._keeps_rows(node):
                    return self._whole_batch(node, v, node.size[1:])
                if fn == "squeeze" and node.attrs["kwargs"].get("dim") == 1 and child.size[1] == 1:
                    return self._whole_batch(node, v, node.size[1:])
                if op == "dropout":
                    twice = any(self._overlap([a], v.segs[:i]) for i, a in enumerate(v.segs))
                    if not twice:  # (rows read twice are drawn for twice)
                        return self._whole_batch(node, v, node.size[1:])
                elif fn in _ROWWISE and self._plain(node):
                    return self._whole_batch(node, v, node.size[1:])
        ins = {k: self._tensor(c) for k, c in node.inputs.items()}
        if op == "call" and node.attrs["fn"] is F.embedding:
            attrs = dict(node.attrs, read_only=all(r.op in ("linear", "typed_linear") for r in
                                                   self.readers.get(id(node), [])) and
                         id(node) not in self.is_root)
            return _Value(ir.Node("call", ins, attrs, node.size))
        return _Value(node.with_inputs(ins))

    @staticmethod
    def _keeps_rows(node):
        args, kw = node.attrs["args"], node.attrs["kwargs"]
        size = kw.get("size", args[1] if len(args) == 2 else args[1:])
        if not isinstance(size, (list, tuple)):
            size = [size]
        return len(size) >= 2 and size[0] in (-1, node.size[0]) and \
            all(isinstance(s, int) for s in size) and isinstance(args[0], ir.Slot)

    @staticmethod
    def _plain(node):
        args, kw = node.attrs["args"], node.attrs["kwargs"]
        return len(args) >= 1 and isinstance(args[0], ir.Slot) and not kw.get("inplace") and \
            all(isinstance(a, (int, float)) for a in args[1:]) and \
            not any(torch.is_tensor(a) for a in kw.values())

    # -- classes of nodes that run together -----------------------------------------------
    def _class_of(self, node):
        if node.op in ("linear", "bundle", "typed_linear"):
            ws = weights_of(node)
            if all(torch.is_tensor(w) and w.dim() == 2 and w.dtype == torch.float32 and
                   w.shape == ws[0][0].shape for w, _ in ws) and \
                    all(c.size is not None and len(c.size) == 2 for c in node.inputs.values()):
                return ("linear",) + tuple(ws[0][0].shape)
        elif node.op == "spmm":
            e = node.inputs.get("e")
            x = self.value.get(id(node.inputs["x"]))
            if x is not None and not x.blocks and len(node.inputs["x"].size) == 3 and \
                    (e is None or (e.op == "edge_values" and e.size[1] == 1 and
                                   node.inputs["x"].size[1] == 1)):
                return ("spmm", id(x.node), e is None) + tuple(node.inputs["x"].size[1:])
        elif node.op == "gat":
            q, k, x = (self.value.get(id(node.inputs[i])) for i in ("q", "k", "x"))
            if q is not None and k is not None and x is not None and k.segs is not None and \
                    x.segs is not None and [n for _, n in k.segs] == [n for _, n in x.segs] and \
                    q.segs is not None and not k.blocks and not x.blocks and \
                    (q.blocks == len(q.segs) if q.blocks else len(q.segs) == 1):
                return ("gat", id(q.node), id(k.node), id(x.node), bool(node.attrs.get("head_mean")))
        return None

    def _count(self, members):
        self.together = self.together or len(members) > 1

    def _linears(self, members):
        units = []  # (query side, node, which, weight, bias, original input)
        for m in members:
            for i, (w, b) in enumerate(weights_of(m)):
                x = m.inputs["x"] if "x" in m.inputs else m.inputs[str(i)]
                side = id(m) in self.query_side
                if m.op == "bundle":
                    side = any(id(r) in self.query_side and r.attrs.get("index") == i
                               for r in self.readers.get(id(m), []))
                units.append((side, m, i, w, b, x))
        units.sort(key=lambda u: not u[0])
        bases, refs = [], []
        for _, _, _, _, _, x in units:
            v = self.value[id(x)]
            segs = _merge(self._segs(v)) if not v.blocks else []
            if len(segs) == 1:
                base, (first, rows) = v.node, segs[0]
            else:
                base = self._tensor(x)
                first, rows = 0, self._rows_of(base)
            at = next((i for i, b in enumerate(bases) if b is base), len(bases))
            if at == len(bases):
                bases.append(base)
            refs.append((at, first, rows))
        m = members[0]
        if len(members) == 1 and (len(units) == 1 or m.op == "bundle") and \
                refs[0][1:] == (0, self._rows_of(bases[0])):
            # nobody to join: a product is a launch, and so are the two of a bundle (with a few
            # outputs a kernel of their own that reads x once)
            self._done(m, _Value(m.with_inputs({k: bases[0] for k in m.inputs})))
            return
        self._count(members)
        self.unit_rows += [rows for _, _, rows in refs]
        made = ir.Node("typed_rows", {str(i): b for i, b in enumerate(bases)},
                       {"units": refs, "weights": [u[3] for u in units], "biases": [u[4] for u in units],
                        "base_rows": [self._rows_of(b) for b in bases]},
                       [sum(r[2] for r in refs), int(units[0][3].size(0))])
        place, off = {}, 0
        for (_, m, i, _, _, _), (_, _, rows) in zip(units, refs):
            place[id(m), i] = (off, rows)
            off += rows
        for m in members:
            own = [place[id(m), i] for i in range(len(weights_of(m)))]
            if m.op == "bundle" or "split" in m.attrs:
                self.parts[id(m)] = [_Value(made, [s]) for s in own]
            self._done(m, _Value(made, own))

    def _chain(self, node):
        """What follows an aggregation on its own: (last node, divisor, act, alpha, row shape)."""
        divisor, tail = 1.0, node.size[1:]
        while True:
            readers = self.readers.get(id(node), [])
            if id(node) in self.is_root or len(readers) != 1 or len(readers[0].inputs) != 1 or \
                    readers[0].size is None:
                return node, divisor, 0, 0.0, tail
            nxt = readers[0]
            fn = nxt.fn_name() if nxt.op == "call" else None
            if fn == "squeeze" and nxt.attrs["kwargs"].get("dim") == 1 and node.size[1] == 1 and \
                    len(node.size) == 3:
                tail = nxt.size[1:]
            elif fn in ("div", "__truediv__", "truediv") and _scalar_call(nxt) and divisor == 1.0:
                divisor = _scalar_call(nxt)
            elif nxt.op == "dropout" and (not self.training or nxt.attrs["p"] == 0):
                pass
            elif fn in _FOLD_ACT and nxt.attrs["fn"] in (F.relu, F.elu, torch.relu) and self._plain(nxt):
                args, kw = nxt.attrs["args"], nxt.attrs["kwargs"]
                alpha = float(kw.get("alpha", args[1] if len(args) > 1 else 1.0))
                if not set(kw) <= {"alpha", "inplace"} or len(args) > 2 or (fn == "elu" and alpha <= 0):
                    return node, divisor, 0, 0.0, tail
                return nxt, divisor, _FOLD_ACT[fn], alpha, nxt.size[1:]
            else:
                return node, divisor, 0, 0.0, tail
            node = nxt

    def _sums(self, members, places):
        """The members, those whose results are only ever added up joined: [(nodes that the sum
        makes unnecessary, its last node, its row ranges in the order of the additions)]."""
        parts = {}  # id of a member's last view -> what stands in the result
        for m, p in zip(members, places):
            through = []
            while len(self.readers.get(id(m), [])) == 1 and id(m) not in self.is_root:
                nxt = self.readers[id(m)][0]
                if not (nxt.op == "call" and nxt.fn_name() == "squeeze" and len(nxt.inputs) == 1 and
                        nxt.attrs["kwargs"].get("dim") == 1 and len(m.size) == 3 and m.size[1] == 1):
                    break
                through.append(m)
                m = nxt
            parts[id(m)] = (through, m, p)
        waiting = list(parts)
        while waiting:
            first = parts.get(waiting.pop())
            if first is None:
                continue
            readers = self.readers.get(id(first[1]), [])
            add = readers[0] if len(readers) == 1 else None
            if add is None or not _is_add(add) or id(first[1]) in self.is_root:
                continue
            a, b = (add.inputs[s.key] for s in add.attrs["args"])
            # a left-hand chain, so that the sum adds in its order; ((a + b) + c)
            if a is b or id(a) not in parts or id(b) not in parts or a.size != b.size or \
                    len(parts[id(b)][2]) != 1 or \
                    any(len(self.readers[id(c)]) != 1 or id(c) in self.is_root for c in (a, b)):
                continue
            (ta, _, pa), (tb, _, pb) = parts.pop(id(a)), parts.pop(id(b))
            parts[id(add)] = (ta + [a] + tb + [b], add, pa + pb)
            waiting.append(id(add))
        return list(parts.values())

    def _fold(self, members, made, places):
        """Values of the members (``places``: the row ranges of each, to be added up)."""
        sums = self._sums(members, places)
        ends = [self._chain(m) for _, m, _ in sums]
        if all(e[1:4] == (1.0, 0, 0.0) and len(p) == 1 for e, (_, _, p) in zip(ends, sums)):
            for m, p in zip(members, places):
                self._done(m, _Value(made, p))
            return
        ranges = [(p[0][1], [o for o, _ in p], d, act, alpha)
                  for (_, d, act, alpha, _), (_, _, p) in zip(ends, sums)]
        off = 0
        groups = {}  # rows of one shape make one value; (they do, but for members of other shapes)
        for e in ends:
            groups.setdefault(tuple(e[4]), None)
        (tail,) = groups if len(groups) == 1 else (tuple(made.size[1:]),)
        node = ir.Node("fold", {"x": made}, {"ranges": ranges, "tail": list(tail)},
                       [sum(r[0] for r in ranges)] + list(tail))
        for (through, m, _), (last, _, _, _, own), r in zip(sums, ends, ranges):
            for n in through:  # the nodes in between exist no longer
                self._finish(n)
            while m is not last:
                self._finish(m)
                m = self.readers[id(m)][0]
            v = _Value(node, [(off, r[0])])
            if tuple(own) != tail:
                v = _Value(ir.Node("call", {"0": self._piece(node, off, r[0])},
                                   {"fn": torch.Tensor.view, "args": (ir.Slot("0"), [-1] + list(own)),
                                    "kwargs": {}}, [r[0]] + list(own)))
            self._done(last, v)
            off += r[0]

    @staticmethod
    def _piece(node, first, rows):
        return ir.Node("rows", {"x": node}, {"first": first, "rows": rows}, [rows] + node.size[1:])

    def _fits(self, members):
        return self._rows_of(self.value[id(members[0].inputs["x"])].node) <= MAX_COLUMNS

    def _alone(self, m):
        ins = {k: self._tensor(c) for k, c in m.inputs.items()}
        self._done(m, _Value(m.with_inputs(ins)))

    def _spmms(self, members):
        xv = [self.value[id(m.inputs["x"])] for m in members]
        if not self._fits(members) or (len(members) == 1 and xv[0].segs is None):
            for m in members:
                self._alone(m)
            return
        self._count(members)
        inputs, spec, places, off = {"x": xv[0].node}, [], [], 0
        for i, (m, x) in enumerate(zip(members, xv)):
            inputs["g%d" % i] = self._tensor(m.inputs["g"])
            scales = []
            if "e" in m.inputs:
                e = m.inputs["e"]
                scales = [e.inputs[str(j)] for j in range(len(e.inputs) - 1)]
                for j, s in enumerate(scales):
                    inputs["s%d.%d" % (i, j)] = self._tensor(s)
            spec.append((self._segs(x), len(scales)))
            rows = int(m.size[0])
            places.append([(off, rows)])
            off += rows
        made = ir.Node("spmm_rows", inputs, {"spec": spec, "n_cols": self._rows_of(xv[0].node)},
                       [off] + members[0].inputs["x"].size[1:])
        self._fold(members, made, places)

    @staticmethod
    def _gathered(node, segs):
        """Row ranges of ``node`` one below the other."""
        return ir.Node("fold", {"x": node}, {"ranges": [(n, [o], 1.0, 0, 0.0) for o, n in segs],
                                             "tail": node.size[1:]},
                       [sum(n for _, n in segs)] + node.size[1:])

    def _keys_of(self, members):
        """{rows of the features: rows of the keys that belong to them}, or None where two members
        put different keys beside the same features or a query feeds two members."""
        pairs, queries = {}, set()
        for m in members:
            ks, xs = self.value[id(m.inputs["k"])].segs, self.value[id(m.inputs["x"])].segs
            if any(pairs.setdefault(x, k) != k for k, x in zip(ks, xs)):
                return None
            for seg in self.value[id(m.inputs["q"])].segs:
                if seg in queries:
                    return None
                queries.add(seg)
        return pairs

    def _keys_beside(self, members, k, x):
        """The node whose rows are the keys in the order of the features' rows."""
        pairs = self._keys_of(members)
        if all(a == b for a, b in pairs.items()) and self._rows_of(k.node) == self._rows_of(x.node):
            return k.node
        ranges, at = [], 0
        for (o, n), (source, _) in sorted(pairs.items()):
            if o > at:
                ranges.append((o - at, [], 1.0, 0, 0.0))
            ranges.append((n, [source], 1.0, 0, 0.0))
            at = o + n
        if at < self._rows_of(x.node):
            ranges.append((self._rows_of(x.node) - at, [], 1.0, 0, 0.0))
        return ir.Node("fold", {"x": k.node}, {"ranges": ranges, "tail": k.node.size[1:]},
                       [self._rows_of(x.node)] + k.node.size[1:])

    def _gats(self, members):
        if not self._fits(members) or self._keys_of(members) is None:
            for m in members:
                self._alone(m)
            return
        self._count(members)
        self.attention = True
        q = self.value[id(members[0].inputs["q"])]
        k = self.value[id(members[0].inputs["k"])]
        x = self.value[id(members[0].inputs["x"])]
        rels = []  # (query rows, member, block)
        for i, m in enumerate(members):
            for b, seg in enumerate(self.value[id(m.inputs["q"])].segs):
                rels.append((seg, i, b))
        rels.sort(key=lambda r: r[0])
        run = _merge([r[0] for r in rels])
        keys = self._keys_beside(members, k, x)
        if len(run) == 1 and q.node is keys:
            query, first = None, run[0][0]  # read where it is
        else:
            query, first = self._gathered(q.node, [r[0] for r in rels]), 0
        inputs = {"k": keys, "x": x.node}
        if query is not None:
            inputs["q"] = query
        for i, m in enumerate(members):
            inputs["g%d" % i] = self._tensor(m.inputs["g"])
        spec = [(i, b, max(1, self.value[id(members[i].inputs["q"])].blocks),
                 self.value[id(members[i].inputs["x"])].segs) for _, i, b in rels]
        places, off = [[] for _ in members], 0
        for (_, n), i, b in rels:
            places[i].append((b, off, n))
            off += n
        places = [[(o, n) for _, o, n in sorted(p)] for p in places]
        mean = bool(members[0].attrs.get("head_mean"))
        made = ir.Node("gat_rows", inputs, {"spec": spec, "first": first, "head_mean": mean,
                                            "n_cols": self._rows_of(x.node)},
                       [off] + x.node.size[2 if mean else 1:])
        self._fold(members, made, places)

    # -- the agenda -------------------------------------------------------------------------
    def _finish(self, node):
        for r in self.readers.get(id(node), []):
            self.pending[id(r)] -= 1
            if self.pending[id(r)] == 0:
                self.ready.append(r)
        self.finished.add(id(node))

    def _done(self, node, value):
        self.value[id(node)] = value
        self._finish(node)

    def build(self):
        self.finished = set()
        self.pending = {id(n): len({id(c) for c in n.inputs.values()}) for n in self.order}
        place = {id(n): i for i, n in enumerate(self.order)}
        self.ready = [n for n in self.order if self.pending[id(n)] == 0]
        waiting = []
        while self.ready or waiting:
            while self.ready:
                n = self.ready.pop()
                if id(n) in self.finished:
                    continue
                if self._class_of(n) is None:
                    self._done(n, self._immediate(n))
                else:
                    waiting.append(n)
            if not waiting:
                break
            classes = {}
            for n in waiting:
                classes.setdefault(self._class_of(n), []).append(n)
            key = min(classes, key=lambda c: sum(self.depth[id(n)] for n in classes[c]) / len(classes[c]))
            members = sorted(classes[key], key=lambda n: place[id(n)])
            taken = {id(n) for n in members}
            waiting = [n for n in waiting if id(n) not in taken]
            {"linear": self._linears, "spmm": self._spmms, "gat": self._gats}[key[0]](members)
        if not self.together or (self.attention and
                                 sum(self.unit_rows) >= MANY_ROWS * len(self.unit_rows)):
            return None
        flow = self._outputs()
        nodes = ir.walk(flow)
        slices = [n for n in nodes if n.op == "rows"]
        ops = sum(bool(n.inputs) for n in self.order) - sum(bool(n.inputs) for n in nodes) + len(slices)
        cut = sum(4 * math.prod(n.inputs["x"].size) for n in slices)
        if cut * CUT_US_PER_BYTE + len(slices) * US_PER_NODE > ops * US_PER_NODE:
            return None
        return flow

    def _outputs(self):
        """The roots. Those that tile one fold become its separate outputs (whose backward takes
        one concatenation of the incoming gradients)."""
        found = {}
        for r in self.roots:
            v = self.value[id(r)]
            if v.node.op == "fold" and v.segs is not None and len(v.segs) == 1 and \
                    len(v.node.size) == 2:
                found.setdefault(id(v.node), (v.node, set()))[1].add(v.segs[0])
        read = {id(c) for n in ir.walk({str(i): self.value[id(r)].node for i, r in enumerate(self.roots)})
                for c in n.inputs.values()}
        splits = {}
        for key, (node, segs) in found.items():
            segs = sorted(segs)
            if len(segs) > 1 and key not in read and _merge(segs) == [(0, self._rows_of(node))]:
                parts = ir.Node("fold", node.inputs, dict(node.attrs, split=[n for _, n in segs]))
                for i, (o, n) in enumerate(segs):
                    splits[key, (o, n)] = ir.Node("select", {"x": parts}, {"index": i},
                                                  [n] + node.size[1:])

        def out(r):
            v = self.value[id(r)]
            hit = splits.get((id(v.node), v.segs[0])) if v.segs else None
            return hit if hit is not None else self._tensor(r)

        if isinstance(self.flow, ir.Node):
            return out(self.flow)
        return {k: out(r) for k, r in self.flow.items()}


def batch_rows(dataflow: ir.Dataflow, kwargs: dict, training: bool = False):
    """The batched form of ``dataflow`` for arguments shaped like ``kwargs`` (outputs and
    gradients as before), or None where nothing runs together, or nothing is gained by it."""
    return _Batcher(dataflow, kwargs, training).build()


# ---- evaluation -------------------------------------------------------------------------
def _columns(blk, segs):
    """Columns of a (possibly stitched) block as rows of the batch that holds its features."""
    cols = blk.adj_sparse[1].to(torch.int64) & mp.COL_MASK
    if len(segs) == 1:
        return cols + segs[0][0]
    dev = cols.device
    ends = torch.tensor([n for _, n in segs], device=dev).cumsum(0)
    shift = torch.tensor([o for o, _ in segs], device=dev)
    shift[1:] -= ends[:-1]
    return cols + shift[torch.bucketize(cols, ends, right=True)]


def _block(indptrs, columns, n_cols):
    """Row-wise stack of CSRs over the same columns."""
    counts = torch.cat([p[1:] - p[:-1] for p in indptrs])
    indptr = torch.zeros(counts.numel() + 1, dtype=torch.int32, device=counts.device)
    indptr[1:] = torch.cumsum(counts, 0)
    return block.Block([counts.numel(), n_cols], [indptr, torch.cat(columns).to(torch.int32)])


def spmm_block(blocks, spec, n_cols):
    return _block([b.adj_sparse[0] for b in blocks],
                  [_columns(b, segs) for b, (segs, _) in zip(blocks, spec)], n_cols)


def gat_block(blocks, spec, n_cols):
    """One row per (relation, destination), relations in the order of ``spec``."""
    indptrs, columns = [], []
    for i, tag, n_blocks, segs in spec:
        b = blocks[i]
        cols = _columns(b, segs)
        if n_blocks == 1:
            indptrs.append(b.adj_sparse[0])
            columns.append(cols)
            continue
        rows, _, tags = mp.edge_endpoints(b)
        own = tags == tag
        indptr = torch.zeros(b.size[0] + 1, dtype=torch.int32, device=cols.device)
        indptr[1:] = torch.cumsum(torch.bincount(rows[own], minlength=b.size[0]), 0)
        indptrs.append(indptr)
        columns.append(cols[own])
    return _block(indptrs, columns, n_cols)
