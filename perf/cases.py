"""The workloads this library is timed on, through its public entry points.

Each listed case stands for one thing a user of the library does: converting a
graph to SWTCF, building the block matrices of a sampled subgraph and
aggregating over them, a product over a graph that is kept, the first layer
over hot and cold feature rows, a GCN training step and its dense products.
`draw` gives more cases of the same kinds over the same ranges, odd and ragged
sizes among them.  Sizes come from tcc_amd.graphs.CONFIGS (graphs of 4,096 to
2.45M nodes, 65k to 114M edges, 32 to 602 features) and, between them, from
the sizes the tests use.  All inputs are seeded and made on the GPU.
"""
from __future__ import annotations

import math
import os
import sys

import torch

from tcc_amd import gcn, graphs, swtcf


# ---------------------------------------------------------------- cases


def listed():
    return [
        # The smallest conversion a caller makes: one small graph (4,096 nodes,
        # 16 sources a row, CSR order), where launches count.
        dict(name="convert_small", kind="convert", graph="uniform", n=4096, edges=65536, S=16, order="rows"),
        # A whole large graph converted once: 233k nodes, 114M edges.
        dict(name="convert_large", kind="convert", graph="rmat", n=233_000, edges=114_000_000, S=16, order="rows"),
        # launchSWTCFSpMM's general form on the small uniform graph.
        dict(name="swtcf_small", kind="swtcf", graph="uniform", n=4096, edges=65536, F=32, S=16),
        # launchSWTCFSpMM's own width on a skewed subgraph of a size that
        # sampling gives, used once or twice.
        dict(name="swtcf_sampled", kind="swtcf", graph="rmat", n=20_000, edges=240_000, F=128, S=16),
        # A product over a kept BCSR with values: 169k nodes, 1.17M edges.
        dict(name="gather_forward", kind="gather", n=169_000, edges=1_170_000, F=128, values=True),
        # A sampled subgraph's layer: both block matrices built from its COO,
        # the forward product and the backward one over Aᵀ.
        dict(name="sampled_layer", kind="layer", n=169_000, edges=1_170_000, F=128),
        # The training scripts' own call: forward_tensorcore over a BCSR and a
        # BCSC part, each feature row gathered often (x is packed first).
        dict(name="extension_forward", kind="extension", n=100_000, edges=3_000_000, F=256, hot=0.5),
        # The largest product over a kept graph: 233k nodes, 114M edges, 602
        # features, symmetric-normalised values as row and column scales.
        dict(name="hybrid_large", kind="hybrid", n=233_000, edges=114_000_000, F=602, build=False),
        # The same kind of graph laid out and multiplied once: what a user
        # waits for before the first result.
        dict(name="hybrid_first_product", kind="hybrid", n=233_000, edges=57_000_000, F=128, build=True),
        # The first layer with 20% of the feature rows in HBM and the rest read
        # from pinned host memory.
        dict(name="mixed_first_layer", kind="mixed", n=2_450_000, edges=61_900_000, F=100, hot=0.2),
        # A full-graph training step of the two-layer GCN (100 -> 256 -> 2) with
        # every feature row in HBM: logits, loss and both weight gradients.
        dict(name="gcn_step", kind="gcn", n=2_450_000, edges=61_900_000, F=100, hidden=256, classes=2),
        # The weight gradient of a wide first layer: 233k nodes, 602 -> 256.
        dict(name="weight_gradient", kind="dense", n=233_000, F=602, hidden=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["convert", "convert", "swtcf", "gather", "layer", "layer", "extension", "hybrid", "mixed", "gcn",
                       "dense"])
    if kind == "convert":
        n = _log_int(rng, 500, 300_000)
        return dict(kind=kind, graph="rmat", n=n, edges=min(20_000_000, int(n * rng.uniform(4, 60))),
                    S=rng.choice([16, 16, 8, 32, 5]), order=rng.choice(["rows", "rows", "shuffled"]))
    if kind == "swtcf":
        n = _log_int(rng, 800, 20_000)
        return dict(kind=kind, graph=rng.choice(["uniform", "rmat"]) if n <= 8000 else "rmat", n=n,
                    edges=n * rng.randint(4, 12), F=_log_int(rng, 16, 256), S=16)
    if kind == "gather":
        n = _log_int(rng, 2_000, 400_000)
        return dict(kind=kind, n=n, edges=int(n * rng.uniform(3, 30)), F=_log_int(rng, 17, 300),
                    values=rng.random() < 0.5)
    if kind == "layer":
        n = _log_int(rng, 1_000, 300_000)
        return dict(kind=kind, n=n, edges=int(n * rng.uniform(3, 25)), F=_log_int(rng, 16, 256))
    if kind == "extension":
        n = _log_int(rng, 5_000, 120_000)
        return dict(kind=kind, n=n, edges=int(n * rng.uniform(10, 40)), F=_log_int(rng, 32, 400),
                    hot=round(rng.uniform(0.2, 1.0), 2))
    if kind == "hybrid":
        n = _log_int(rng, 20_000, 200_000)
        return dict(kind=kind, n=n, edges=int(n * rng.uniform(100, 300)), F=_log_int(rng, 32, 600),
                    build=rng.random() < 0.5)
    if kind == "mixed":
        n = _log_int(rng, 20_000, 800_000)
        return dict(kind=kind, n=n, edges=int(n * rng.uniform(6, 25)), F=_log_int(rng, 20, 128),
                    hot=round(rng.uniform(0.1, 0.9), 2))
    if kind == "gcn":
        n = _log_int(rng, 3_000, 1_000_000)
        return dict(kind=kind, n=n, edges=int(n * rng.uniform(4, 25)), F=_log_int(rng, 16, 128),
                    hidden=rng.choice([16, 64, 128, 200, 256]), classes=rng.randint(2, 8))
    return dict(kind="dense", n=_log_int(rng, 10_000, 2_000_000), F=_log_int(rng, 16, 300),
                hidden=_log_int(rng, 2, 256))


# ---------------------------------------------------------------- inputs


class _DeviceArray:
    """Device memory at an address, as torch.as_tensor takes it (no copy)."""

    def __init__(self, ptr, count, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(int(count),), typestr=typestr, data=(int(ptr), False), version=2)


def _view(ptr, count, typestr, owner):
    return torch.as_tensor(_DeviceArray(ptr, count, typestr, owner), device="cuda")


def _uniform(n, deg, seed):
    """Every row gets `deg` distinct uniform columns, in (row, column) order."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    cols = torch.topk(torch.rand((n, n), generator=g, device="cuda"), deg, dim=1).indices
    cols = torch.sort(cols, dim=1).values
    rows = torch.arange(n, device="cuda").repeat_interleave(deg)
    return rows, cols.reshape(-1)


def _edges(case, seed):
    """(rows, cols) int64 in (row, column) order."""
    n, edges = case["n"], case["edges"]
    if case.get("graph") == "uniform":
        return _uniform(n, edges // n, seed)
    return graphs.rmat_graph(n, edges, seed, device="cuda")


def _normal(rows, cols, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn((rows, cols), generator=g, device="cuda")


def _extension():
    """The spmm_cnic module, imported as the training scripts import it."""
    where = os.path.join(os.path.dirname(os.path.abspath(swtcf.__file__)))
    if where not in sys.path:
        sys.path.insert(0, where)
    import spmm_cnic

    return spmm_cnic


def _block_args(view, kind, owner):
    """A block matrix's arrays as the extension's arguments."""
    if kind == "bcsr":
        windows, offset, idx = view.num_rowWindows, view.rowWindowOffset, view.sparseA2B
    else:
        windows, offset, idx = view.num_colWindows, view.colWindowOffset, view.sparseA2C
    B = view.num_TCBlocks
    return [view.num_rows, view.num_cols, view.nnz, B, windows, _view(offset, windows + 1, "<i4", owner),
            _view(view.tcOffset, B + 1, "<i4", owner), _view(idx, 8 * B, "<i4", owner),
            _view(view.tcLocalBit, B, "<i8", owner), torch.zeros(1, device="cuda")]


def _swtcf_views(m, n, edges):
    """The arrays of a conversion of `edges` edges, the tile and row arrays up
    to what any such graph can fill, cleared once."""
    v = m.m
    cols_windows, super_windows = m.numColWindows, m.numSuperWindows
    tiles, rows = min(edges, edges // 8 + cols_windows), min(edges, n * super_windows)
    out = dict(
        colWindowOffset=_view(v.colWindowOffset, cols_windows + 1, "<i4", m),
        superWindowRowOffset=_view(v.superWindowRowOffset, super_windows + 1, "<i4", m),
        tileLocalBit=_view(v.tileLocalBit, tiles, "<i8", m),
        tileRowSlot=_view(v.tileRowSlot, 8 * tiles, "<i4", m),
        superWindowRows=_view(v.superWindowRows, rows, "<i4", m),
        superWindowRowCacheSlot=_view(v.superWindowRowCacheSlot, rows, "|u1", m),
        superWindowCachedRowSlot=_view(v.superWindowCachedRowSlot, 32 * super_windows, "<i4", m),
        superWindowCachedCount=_view(v.superWindowCachedCount, super_windows, "|u1", m),
    )
    for t in out.values():
        t.zero_()
    return out


def _i32(t):
    return t.to(torch.int32).contiguous()


# ---------------------------------------------------------------- prepare / run


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dense":
        return dict(case=case, A=_normal(case["n"], case["F"], seed + 1), B=_normal(case["n"], case["hidden"], seed + 2))
    n = case["n"]
    rows, cols = _edges(case, seed)
    s = dict(case=case)
    if kind == "convert":
        S = case["S"]
        if case["order"] == "shuffled":
            g = torch.Generator(device="cuda").manual_seed(seed + 3)
            p = torch.randperm(rows.numel(), generator=g, device="cuda")
            rows, cols = rows[p], cols[p]
        s["dst"], s["src"] = _i32(rows), _i32(cols)
        s["m"] = swtcf.DeviceSWTCFMatrix(n, n, rows.numel(), S)
        s["ws"] = swtcf.SWTCFConvertWorkspace(rows.numel(), n, S)
        s["out"] = _swtcf_views(s["m"], n, rows.numel())
        return s
    F = case["F"]
    if kind == "swtcf":
        s["m"] = swtcf.DeviceSWTCFMatrix(n, n, rows.numel(), case["S"])
        ws = swtcf.SWTCFConvertWorkspace(rows.numel(), n, case["S"])
        swtcf.convertCOOToSWTCF(_i32(rows), _i32(cols), rows.numel(), s["m"], ws)
        if ws.device_error() != 0:
            raise RuntimeError("conversion failed")
        s["X"] = _normal(n, F, seed + 1)
        s["Y"] = torch.zeros((n, F), device="cuda")
    elif kind == "gather":
        vals = graphs.sym_norm_values(rows, cols, n) if case["values"] else None
        s["A"] = swtcf.coo_to_bcsr(_i32(rows), _i32(cols), vals, n, n)
        s["X"] = _normal(n, F, seed + 1)
        s["Y"] = torch.empty((s["A"].out_windows * 8, F), device="cuda")
    elif kind == "layer":
        s["rows"], s["cols"] = _i32(rows), _i32(cols)
        s["X"], s["dY"] = _normal(n, F, seed + 1), _normal(n, F, seed + 2)
    elif kind == "extension":
        g = torch.Generator(device="cuda").manual_seed(seed + 3)
        hot = torch.rand(n, generator=g, device="cuda") < case["hot"]
        h = hot[cols]
        s["A"] = swtcf.coo_to_bcsr(_i32(rows[h]), _i32(cols[h]), None, n, n)
        s["B"] = swtcf.coo_to_bcsc(_i32(rows[~h]), _i32(cols[~h]), None, n, n)
        s["args"] = _block_args(s["A"].view, "bcsr", s["A"]) + _block_args(s["B"].view, "bcsc", s["B"])
        s["x"] = _normal(n, F, seed + 1).reshape(-1)
        s["module"] = _extension()
    elif kind == "hybrid":
        s["r"], s["c"] = graphs.sym_norm_scales(rows, cols, n)
        s["X"] = _normal(n, F, seed + 1)
        s["rows"], s["cols"] = _i32(rows), _i32(cols)
        if not case["build"]:
            s["H"] = _lay_out(s)
            del s["rows"], s["cols"]
            s["Y"] = torch.empty((s["H"].out_rows, F), device="cuda")
            s["workspace"] = torch.empty(s["H"].workspace_bytes(F) + 16, dtype=torch.uint8, device="cuda")
    elif kind in ("mixed", "gcn"):
        X = _normal(n, F, seed + 1)
        s["table"] = gcn.FeatureTable(X, cols, hot_fraction=case.get("hot", 1.0))
        if kind == "mixed":
            s["graph"] = gcn.LayerGraph(rows, cols, n, n, hot_src=s["table"].hot, backward_bcsc=gcn._EMPTY_BCSC)
        else:
            s["g1"], s["g2"] = gcn.build_gcn_graphs(rows, cols, n, s["table"].hot)
            g = torch.Generator(device="cuda").manual_seed(seed + 4)
            s["labels"] = torch.randint(0, case["classes"], (n,), generator=g, device="cuda")
            s["model"] = gcn.GCN(F, case["hidden"], case["classes"], dropout=0.0).cuda()
            with torch.no_grad():
                for k, w in enumerate(_weights(case, seed)):
                    list(s["model"].parameters())[k].copy_(w)
    else:
        raise ValueError(kind)
    return s


def _weights(case, seed):
    """The two layers' weights, xavier-uniform."""
    out = []
    for k, (a, b) in enumerate(((case["F"], case["hidden"]), (case["hidden"], case["classes"]))):
        g = torch.Generator(device="cuda").manual_seed(seed + 5 + k)
        bound = math.sqrt(6.0 / (a + b))
        out.append((torch.rand((a, b), generator=g, device="cuda") * 2 - 1) * bound)
    return out


def _lay_out(s):
    n = s["case"]["n"]
    return swtcf.coo_to_hybrid_scaled(s["rows"], s["cols"], n, n, s["r"], s["c"], phases=2)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "convert":
        swtcf.convertCOOToSWTCF(s["dst"], s["src"], s["dst"].numel(), s["m"], s["ws"])
        return s["out"]
    if kind == "swtcf":
        s["Y"].zero_()
        if case["F"] == swtcf.FEATURE_DIM and case["S"] == 16:
            swtcf.launchSWTCFSpMM(s["m"], s["X"], s["Y"])
        else:
            swtcf.swtcf_spmm(s["m"], s["X"], s["Y"])
        return s["Y"]
    if kind == "gather":
        return swtcf.bcsr_spmm(s["A"], s["X"], s["Y"])
    if kind == "layer":
        n = case["n"]
        graph = gcn.LayerGraph(s["rows"], s["cols"], n, n)
        return graph.aggregate(case["F"], x=s["X"]), graph.transpose_aggregate(s["dY"])
    if kind == "extension":
        out = s["module"].forward_tensorcore(*s["args"], case["F"], s["x"])
        s["module"].freeMatC()
        return out.reshape(case["n"], case["F"])
    if kind == "hybrid":
        if case["build"]:
            return swtcf.hybrid_spmm(_lay_out(s), s["X"])[: case["n"]]
        return swtcf.hybrid_spmm(s["H"], s["X"], s["Y"], workspace=s["workspace"])[: case["n"]]
    if kind == "mixed":
        return s["graph"].aggregate(case["F"], source=s["table"].source)
    if kind == "gcn":
        model = s["model"]
        model.zero_grad()
        logits = model(s["g1"], s["g2"], s["table"].source)
        loss = gcn.cross_entropy(logits, s["labels"])
        loss.backward()
        return dict(logits=logits.detach(), loss=loss.detach(), grads=[p.grad for p in model.parameters()])
    return swtcf.dense_tn(s["A"], s["B"])


# ---------------------------------------------------------------- figures


def work(case):
    """Inputs read once and outputs written once."""
    kind, n = case["kind"], case["n"]
    if kind == "dense":
        F, hid = case["F"], case["hidden"]
        return {"bytes": 4 * (n * (F + hid) + F * hid), "flops": 2 * n * F * hid}
    e = case["edges"]
    if kind == "convert":
        # the COO; per (window, row) group, of which these graphs have about
        # one an edge, a slot and a bitmap byte; per row of a super-window,
        # at least one for every 8 edges, its id and its cache slot
        return {"bytes": 8 * e + 5 * e + 5 * (e // 8), "flops": 0}
    F = case["F"]
    rows = 4 * F * n
    # a block matrix holds at least a row index an edge and 12 bytes a block of 8
    blocks = 4 * e + 12 * (e // 8) + 4 * (n // 8 + 1)
    if kind == "swtcf":
        return {"bytes": 2 * rows + 5 * e + 5 * (e // 8), "flops": 2 * e * F}
    if kind == "gather":
        return {"bytes": 2 * rows + blocks + (4 * e if case["values"] else 0), "flops": 2 * e * F}
    if kind == "layer":
        return {"bytes": 4 * rows + 8 * e + 2 * blocks, "flops": 4 * e * F}
    if kind == "hybrid":
        read = 8 * e if case["build"] else 4 * e
        return {"bytes": 2 * rows + read + 8 * n, "flops": 2 * e * F}
    if kind == "gcn":
        h, c = case["hidden"], case["classes"]
        # X and AX, H and its products, and the class-width products over A and Aᵀ
        return {"bytes": 3 * blocks + rows * 3 + 4 * n * (2 * h + 6 * c + 2),
                "flops": 2 * e * (F + 2 * c) + 4 * n * F * h + 6 * n * h * c}
    return {"bytes": 2 * rows + blocks, "flops": 2 * e * F}


def tolerance(case):
    if case["kind"] == "convert":
        return "exact"
    if case["kind"] == "gcn":
        # gradients: sums over every node of rounded products
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 5e-6, "max": 2e-4}


# ---------------------------------------------------------------- 64 bits


def _product(rows, cols, X, n, vals=None):
    """Y[n x F] = A X in float64; edges (rows, cols) with values or ones."""
    X = X.double()
    Y = torch.zeros((n, X.shape[1]), dtype=torch.float64, device=X.device)
    step = max(1, (1 << 29) // X.shape[1])
    for e in range(0, rows.numel(), step):
        part = X[cols[e:e + step]]
        if vals is not None:
            part *= vals[e:e + step].double().unsqueeze(1)
        Y.index_add_(0, rows[e:e + step], part)
    return Y


def exact(case, seed):
    """What run() returns, in float64, from plain torch."""
    kind = case["kind"]
    if kind == "convert":
        return None  # whole numbers
    if kind == "dense":
        A, B = _normal(case["n"], case["F"], seed + 1), _normal(case["n"], case["hidden"], seed + 2)
        out = torch.zeros((case["F"], case["hidden"]), dtype=torch.float64, device="cuda")
        for k in range(0, case["n"], 1 << 18):
            out += A[k:k + (1 << 18)].double().t().contiguous() @ B[k:k + (1 << 18)].double()
        return out
    n, F = case["n"], case["F"]
    rows, cols = _edges(case, seed)
    X = _normal(n, F, seed + 1)
    if kind in ("swtcf", "extension", "mixed"):
        return _product(rows, cols, X, n)
    if kind == "gather":
        Y = _product(rows, cols, X, n, _sym_norm(rows, cols, n) if case["values"] else None)
        return torch.nn.functional.pad(Y, (0, 0, 0, (-n) % 8))
    if kind == "layer":
        return _product(rows, cols, X, n), _product(cols, rows, _normal(n, F, seed + 2), n)
    if kind == "hybrid":
        r, c = (1.0 / torch.sqrt(torch.bincount(i, minlength=n).double().clamp_min(1)) for i in (rows, cols))
        return _product(rows, cols, X.double() * c.unsqueeze(1), n) * r.unsqueeze(1)
    # the GCN step, its gradients written out
    g = torch.Generator(device="cuda").manual_seed(seed + 4)
    labels = torch.randint(0, case["classes"], (n,), generator=g, device="cuda")
    w1, w2 = (w.double() for w in _weights(case, seed))
    AX = _product(rows, cols, X, n)
    H = torch.relu(AX @ w1)
    logits = _product(rows, cols, H @ w2, n)
    p = torch.softmax(logits, dim=1)
    loss = -torch.log_softmax(logits, dim=1).gather(1, labels.view(-1, 1)).mean()
    p[torch.arange(n, device="cuda"), labels] -= 1.0
    G = _product(cols, rows, p / n, n)
    dH = (G @ w2.t()) * (H > 0)
    return dict(logits=logits, loss=loss, grads=[AX.t().contiguous() @ dH, H.t().contiguous() @ G])


def _sym_norm(rows, cols, n):
    """1 / sqrt(row degree * column degree) of each edge, in float64."""
    rd, cd = torch.bincount(rows, minlength=n).double(), torch.bincount(cols, minlength=n).double()
    return 1.0 / torch.sqrt(rd[rows] * cd[cols])
