"""The work that users of this package have it do, as measurable cases: graph preparation, the layers and stand-alone operators,
forward passes and whole training steps (forward, loss, backward) of the three model families of the package's drivers.

Graphs are seeded and have the node and edge counts of the data sets named in `ae_mlsys_gnn_amd.train.datasets.SHAPES`, or those
of the benchmark.  `graph` names their structure: "rmat" (the generator's own labels, where hubs sit at ids with few bits set),
"rmat_permuted" (hubs at arbitrary ids, as in collected data) or "uniform" (no hubs, as in meshes and k-regular graphs)."""
from __future__ import annotations

import math

import torch

from ae_mlsys_gnn_amd import graphs
from ae_mlsys_gnn_amd.layers import EdgeConv, GATConv, GATConv_fusescatter, GATConv_stash, GMMConv, GMMConv_stash
from ae_mlsys_gnn_amd.operators.csr2csc import coo2csr, csr2csc
from ae_mlsys_gnn_amd.operators.fused_gat import fused_gat_operator_pipeline
from ae_mlsys_gnn_amd.operators.knn import knn_graph
from ae_mlsys_gnn_amd.train import common, datasets, train_edgeconv, train_gatconv, train_gmmconv

GAT_CONVS = {"recompute": GATConv, "stash": GATConv_stash, "fusescatter": GATConv_fusescatter}
GMM_CONVS = {"recompute": GMMConv, "stash": GMMConv_stash}
SLOPE = 0.2
DGCNN_WIDTHS = [64, 64, 128, 256]
DGCNN_EMB = [512, 512, 256]


def listed():
    return [
        # one attention layer on a small uniform graph: launches and host work count
        dict(name="gat_layer_small", path="gat_layer", graph="uniform", n=4096, e=32768, fin=64, heads=4, fout=16, variant="recompute"),
        # a citation graph's training step (the drivers' default data set): few edges, 1433 input features
        dict(name="gat_train_cora", path="gat_train", graph="rmat_permuted", n=2708, e=10556, fin=1433, heads=1, fout=128, classes=7,
             variant="recompute"),
        # the benchmark's layer: 115 M edges, degree 490
        dict(name="gat_layer_reddit", path="gat_layer", graph="rmat", n=232965, e=114600000, fin=256, heads=8, fout=32, variant="recompute"),
        # the benchmark's two-layer training step: 2.4 M nodes, features larger than the caches, 47 classes
        dict(name="gat_train_products", path="gat_train", graph="rmat_permuted", n=2449029, e=61859140, fin=100, heads=8, fout=32, classes=47,
             variant="recompute"),
        # a graph in between with the stashing variant
        dict(name="gat_train_arxiv_stash", path="gat_train", graph="rmat_permuted", n=169343, e=2315598, fin=128, heads=4, fout=64, classes=40,
             variant="stash"),
        # inference: one layer forward without gradients, the forward-latency driver's shape
        dict(name="gat_forward_reddit", path="gat_forward", graph="rmat_permuted", n=232965, e=114600000, fin=64, heads=4, fout=64,
             variant="recompute"),
        # the benchmark's mixture-model layer with pseudo-coordinate gradients
        dict(name="gmm_layer_arxiv", path="gmm_layer", graph="rmat", n=169343, e=2315598, fin=128, kernels=3, dim=2, fout=64, variant="recompute"),
        # MoNet training at the largest edge count, narrow rows
        dict(name="monet_train_reddit", path="monet_train", graph="rmat_permuted", n=232965, e=114600000, fin=602, hidden=16, kernels=2, dim=1,
             classes=41, variant="recompute"),
        # two EdgeConv layers with their neighbour graphs on the benchmark's point clouds
        dict(name="edgeconv_stack", path="edgeconv", clouds=32, points=1024, k=20, widths="3,64,64"),
        # a whole point-cloud classifier at the driver's default batch, four neighbour graphs among it, evaluated without gradients (its
        # training step is not a case: chains of maxima and neighbours in feature space flip at near-ties, and its gradients with them)
        dict(name="dgcnn_forward", path="dgcnn_forward", clouds=64, points=1024, k=40, classes=40),
        # attention from the stand-alone per-edge operators, each with its own backward
        dict(name="edge_ops_arxiv", path="edge_ops", graph="rmat_permuted", n=169343, e=2315598, heads=8, fout=32),
        # an unsorted edge list to CSR and CSC, the preparation every graph goes through
        dict(name="graph_build_products", path="graph_build", graph="rmat_permuted", n=2449029, e=61859140),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_graph(rng, max_edges, n_hi=2449029):
    n = _log(rng, 1500, n_hi)
    mean = math.exp(rng.uniform(math.log(3), math.log(490)))
    return dict(graph=rng.choice(["rmat", "rmat_permuted", "rmat_permuted", "uniform"]), n=n, e=max(n, int(min(n * mean, n * (n // 32), max_edges))))


def draw(rng):
    """One more case: any path, sizes spread over their logarithm, odd widths and class counts among them.  The edge count is
    bounded so that rows x width stay within the largest listed case of the path."""
    path = rng.choice(["gat_layer", "gat_train", "gat_forward", "gmm_layer", "monet_train", "edgeconv", "dgcnn_forward", "edge_ops", "graph_build"])
    if path in ("gat_layer", "gat_train", "gat_forward"):
        heads, fout = rng.choice([(8, 32), (4, 64), (4, 16), (8, 8), (1, 128), (2, 30), (1, 41), (3, 20), (6, 64)])
        width = heads * fout
        limit = {"gat_layer": 114600000 * 256, "gat_train": 61859140 * 256, "gat_forward": 114600000 * 256}[path] // max(width, 128)
        c = dict(path=path, **_draw_graph(rng, min(limit, 114600000), n_hi=2449029 if path == "gat_train" else 1000000), fin=_log(rng, 16, 602),
                 heads=heads, fout=fout)
        c["fin"] = min(c["fin"], max(16, 2449029 * 100 // c["n"]))
        if path == "gat_train":
            c["classes"] = rng.randint(3, 50)
        c["variant"] = "recompute" if path == "gat_forward" else rng.choice(["recompute", "recompute", "stash", "fusescatter"])
        if c["variant"] != "recompute":
            c["e"] = max(c["n"], min(c["e"], 30000000))
        return c
    if path == "gmm_layer":
        return dict(path=path, **_draw_graph(rng, 20000000, n_hi=300000), fin=_log(rng, 16, 256), kernels=rng.choice([1, 2, 3]), dim=rng.choice([1, 2, 3]),
                    fout=rng.choice([16, 32, 41, 64]), variant=rng.choice(["recompute", "recompute", "stash"]))
    if path == "monet_train":
        k, dim = rng.choice([(2, 1), (3, 2), (3, 3)])
        return dict(path=path, **_draw_graph(rng, 60000000, n_hi=500000), fin=_log(rng, 16, 602), hidden=rng.choice([16, 16, 32]), kernels=k, dim=dim,
                    classes=rng.randint(3, 47), variant=rng.choice(["recompute", "recompute", "stash"]))
    if path in ("edgeconv", "dgcnn_forward"):
        c = dict(path=path, clouds=_log(rng, 2, 64), points=rng.choice([256, 500, 512, 777, 1024, 1024]), k=rng.choice([5, 10, 20, 20, 30, 40]))
        return dict(c, widths=rng.choice(["3,64,64", "3,32", "6,64,128", "3,40,64"])) if path == "edgeconv" else dict(c, classes=rng.randint(10, 40))
    if path == "edge_ops":
        heads, fout = rng.choice([(8, 32), (4, 16), (1, 64), (2, 30), (4, 64)])
        return dict(path=path, **_draw_graph(rng, 20000000, n_hi=1000000), heads=heads, fout=fout)
    return dict(path=path, **_draw_graph(rng, 61859140))


# ---------------------------------------------------------------- inputs

def _gen(seed, dev):
    return torch.Generator(device=dev).manual_seed(int(seed) * 7919 + 13)


def _make_csr(case, seed, dev):
    """CSR by destination with one self-loop per node; parallel edges merged."""
    n, e = case["n"], case["e"]
    if case["graph"] == "uniform":
        gen = _gen(seed, dev)
        keys = torch.randint(0, n * n, (e + e // 8 + 1024,), generator=gen, device=dev, dtype=torch.int64)
        keys = torch.unique(keys[torch.div(keys, n, rounding_mode="floor") != keys % n])
        keys = keys[torch.randperm(keys.numel(), generator=gen, device=dev)[:e]]
        return graphs.csr_from_keys(graphs.with_self_loops(keys, n), n)
    return graphs.rmat_graph(n, e, seed=int(seed), device=dev, permute_labels=case["graph"] == "rmat_permuted")


def _make_graph(case, seed, dev):
    g = _make_csr(case, seed, dev)
    g.col_ptr, g.row_ind, g.permute = csr2csc(g.row_ptr, g.col_ind)
    return g


def _normal(gen, *shape):
    return torch.randn(*shape, generator=gen, device=gen.device)


def _clouds(gen, b, p):
    """Points on spheres and cubes and inside boxes, scaled per cloud and axis: objects that differ from one another, as in a
    shape classification set."""
    dev = gen.device
    ball = _normal(gen, b, p, 3)
    ball = ball / ball.norm(dim=2, keepdim=True)
    box = torch.rand(b, p, 3, generator=gen, device=dev) * 2 - 1
    axis = torch.randint(0, 3, (b, p, 1), generator=gen, device=dev)
    side = torch.randint(0, 2, (b, p, 1), generator=gen, device=dev).float() * 2 - 1
    kind = torch.randint(0, 3, (b, 1, 1), generator=gen, device=dev)
    return torch.where(kind == 0, ball, torch.where(kind == 1, box.scatter(2, axis, side), box)) * torch.exp(0.5 * _normal(gen, b, 1, 3))


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = _gen(seed, dev)
    torch.manual_seed(int(seed))                # the modules' own initialisation
    s = dict(case=case, path=case["path"])
    path = case["path"]
    if path in ("edgeconv", "dgcnn_forward"):
        b, p = case["clouds"], case["points"]
        if path == "edgeconv":
            widths = [int(w) for w in case["widths"].split(",")]
            s["x"] = torch.rand(b, p, widths[0], generator=gen, device=dev) * 2 - 1
            s["layers"] = [EdgeConv(a, o).to(dev) for a, o in zip(widths, widths[1:])]
            s["params"] = [q for m in s["layers"] for q in m.parameters()]
            s["grad"] = _normal(gen, b * p, widths[-1])
        else:
            s["x"] = _clouds(gen, b, p)
            s["model"] = train_edgeconv.Model(case["k"], DGCNN_WIDTHS, DGCNN_EMB, case["classes"]).to(dev).eval()
        return s
    if path == "graph_build":
        g = _make_csr(case, seed, dev)
        dst = torch.repeat_interleave(torch.arange(g.n, device=dev, dtype=torch.int32), (g.row_ptr[1:] - g.row_ptr[:-1]).long())
        order = torch.randperm(dst.numel(), generator=gen, device=dev)
        s["dst"], s["src"] = dst[order], g.col_ind[order]
        return s
    g = s["g"] = _make_graph(case, seed, dev)
    n = g.n
    if path == "edge_ops":
        h, f = case["heads"], case["fout"]
        s["args"] = [t.requires_grad_(True) for t in (_normal(gen, n, h), _normal(gen, n, h), _normal(gen, n, h, f))]
        s["grad"] = _normal(gen, n, h, f)
        return s
    s["x"] = _normal(gen, n, case["fin"])
    if path in ("gat_layer", "gat_forward"):
        s["layer"] = GAT_CONVS[case["variant"]](case["fin"], case["fout"], case["heads"], SLOPE).to(dev)
        s["extra"] = True if case["variant"] == "recompute" else g.permute
        if path == "gat_layer":
            s["params"] = list(s["layer"].parameters())
            s["grad"] = _normal(gen, n, case["heads"], case["fout"])
        return s
    if path == "gmm_layer":
        s["layer"] = GMM_CONVS[case["variant"]](case["fin"], case["fout"], case["dim"], case["kernels"]).to(dev)
        # what a driver hands the layer: coordinates from the degrees through a small projection, which wants their gradient
        w = _normal(gen, 2, case["dim"])
        s["pseudo"] = torch.tanh(datasets.degree_pseudo(g) @ w).contiguous().requires_grad_(True)
        s["params"] = list(s["layer"].parameters()) + [s["pseudo"]]
        s["grad"] = _normal(gen, n, case["fout"])
        return s
    label = torch.randint(0, case["classes"], (n,), generator=gen, device=dev)
    s["rows"] = common.MaskedRows(torch.rand(n, generator=gen, device=dev) < 0.65, label)
    if path == "gat_train":
        s["model"] = train_gatconv.GAT(GAT_CONVS[case["variant"]], 1, case["fin"], case["fout"], case["classes"], [case["heads"], 1], SLOPE).to(dev)
        s["extra"] = True if case["variant"] == "recompute" else g.permute
    else:
        # the driver's default: the constant edge coordinates in the order in which each pass walks the edges
        s["pseudo"], s["pseudo_csc"] = train_gmmconv.schedule_order_copies(g, datasets.degree_pseudo(g))
        s["model"] = train_gmmconv.MoNet(GMM_CONVS[case["variant"]], case["fin"], case["hidden"], case["classes"], 0, case["dim"], case["kernels"],
                                         0.0).to(dev).train()
    s["params"] = list(s["model"].parameters())
    return s


# ---------------------------------------------------------------- passes

def _with_grads(params, **outs):
    outs["grads"] = [p.grad for p in params]
    return {k: (v.detach() if isinstance(v, torch.Tensor) else v) for k, v in outs.items()}


def run(s):
    path, case = s["path"], s["case"]
    if path == "graph_build":
        row_ptr, col_ind = coo2csr(s["dst"], s["src"], case["n"])
        return (row_ptr, col_ind) + tuple(csr2csc(row_ptr, col_ind))
    if path == "dgcnn_forward":
        with torch.no_grad():
            return s["model"](s["x"])
    if path == "gat_forward":
        g = s["g"]
        with torch.no_grad():
            return s["layer"](g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, s["x"], s["extra"])
    params = s["args"] if path == "edge_ops" else s["params"]
    for p in params:
        p.grad = None
    if path == "edgeconv":
        b, p, _ = s["x"].shape
        h = s["x"]
        for layer in s["layers"]:
            src = knn_graph(h.detach(), case["k"])
            h = layer(case["k"], src, h.reshape(b * p, -1), block=p, negative_slope_out=SLOPE).view(b, p, -1)
        out = h.view(b * p, -1)
        out.backward(s["grad"])
        return _with_grads(params, out=out)
    g = s["g"]
    if path == "edge_ops":
        ar, ac, h = params
        out = fused_gat_operator_pipeline(ar, ac, g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, SLOPE, h, g.permute)
        out.backward(s["grad"])
        return _with_grads(params, out=out)
    if path == "gat_layer":
        out = s["layer"](g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, s["x"], s["extra"])
        out.backward(s["grad"])
        return _with_grads(params, out=out)
    if path == "gmm_layer":
        out = s["layer"](g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, g.permute, s["x"], s["pseudo"])
        out.backward(s["grad"])
        return _with_grads(params, out=out)
    if path == "gat_train":
        logits = s["model"](g, s["x"], s["extra"], keep_padding=True)
        loss = common.masked_cross_entropy(logits, s["rows"], case["classes"])
        logits = logits[:, :case["classes"]]
    else:
        logits = s["model"](g, s["x"], s["pseudo"], s["pseudo_csc"], own_order=True)
        loss = common.masked_cross_entropy(logits, s["rows"])
    loss.backward()
    return _with_grads(params, logits=logits, loss=loss)


# ---------------------------------------------------------------- what a pass cannot do without

def _dense(n, fin, fout, passes):
    """An n-row product with a [fin, fout] weight: the forward, and in training the weight (and input) gradient."""
    return 2.0 * n * fin * fout * passes


def work(case):
    path = case["path"]
    if path in ("edgeconv", "dgcnn_forward"):
        nodes, k, p = case["clouds"] * case["points"], case["k"], case["points"]
        train = path == "edgeconv"
        widths = [int(w) for w in case["widths"].split(",")] if train else [3] + DGCNN_WIDTHS
        flops = by = 0.0
        for i, (a, o) in enumerate(zip(widths, widths[1:])):
            # distances, the two projections (and their gradients), the maxima
            flops += 3.0 * nodes * p * a + _dense(nodes, a, 2 * o, (2 if i == 0 else 3) if train else 1) + (2.0 if train else 1.0) * nodes * k * o
            by += 4.0 * nodes * (a + (2 if train else 1) * o)
        if not train:
            flops += _dense(nodes, sum(DGCNN_WIDTHS), DGCNN_EMB[0], 1)
            by += 4.0 * nodes * sum(DGCNN_WIDTHS)
        return {"bytes": by, "flops": flops}
    n, e = case["n"], case["e"] + case["n"]
    if path == "graph_build":
        return {"bytes": 8.0 * e + 12.0 * e + 8.0 * n, "flops": 0.0}
    if path == "edge_ops":
        hf = case["heads"] * case["fout"]
        return {"bytes": 4.0 * (4 * n * hf + 4 * n * case["heads"] + 3 * e + 2 * n), "flops": 6.0 * e * hf}
    fin = case["fin"]
    if path in ("gat_layer", "gat_forward", "gat_train"):
        hf = case["heads"] * case["fout"]
        fwd = dict(bytes=4.0 * (n * fin + n * hf + e + n), flops=_dense(n, fin, hf, 1) + 2.0 * e * hf)
        if path == "gat_forward":
            return fwd
        layer = dict(bytes=fwd["bytes"] + 4.0 * (n * hf + e + n), flops=fwd["flops"] + _dense(n, fin, hf, 1) + 4.0 * e * hf)
        if path == "gat_layer":
            return layer
        c = case["classes"]
        return {"bytes": layer["bytes"] + 4.0 * n * c, "flops": layer["flops"] + _dense(n, hf, c, 3) + 6.0 * e * c}
    if path == "gmm_layer":
        kf = case["kernels"] * case["fout"]
        return {"bytes": 4.0 * (n * fin + 2 * n * case["fout"] + 2 * e + 2 * n + 2 * e * case["dim"]), "flops": _dense(n, fin, kf, 2) + 6.0 * e * kf}
    k, hid, c = case["kernels"], case["hidden"], case["classes"]
    return {"bytes": 4.0 * (n * fin + n * c + 2 * e + 2 * n + 2 * 2 * e), "flops": _dense(n, fin, k * hid, 2) + 6.0 * e * k * hid
            + _dense(n, k * hid, c, 3) + 6.0 * e * k * hid}


def tolerance(case):
    """About four times what a random change of every input and weight by up to one unit in the last place does to the outputs
    (worst output of each path over sizes drawn from its whole range)."""
    path = case["path"]
    if path == "graph_build":
        return "exact"
    if path == "dgcnn_forward":
        return {"rel": 1.2e-4, "max": 4e-3}         # 3e-5 and 4e-4 seen; 1e-3 in larger batches: a neighbour in feature space that flips at a near-tie
    if path == "edgeconv":
        # flips at near-ties: of the maxima (9e-4 seen), with a second layer of its neighbours too (5e-3)
        return {"rel": 4e-3 if case["widths"].count(",") == 1 else 2e-2, "max": 0.9}
    if path in ("gat_layer", "gat_train"):
        return {"rel": 7e-3, "max": 3e-2}           # 2e-3 and 7e-3 seen: score-weight gradients, cancelling sums with LeakyReLU's jump at 0
    if path == "edge_ops":
        return {"rel": 1e-3, "max": 0.9}            # 2e-4 and 0.4 seen: the same jump in the gradients of single scores
    return {"rel": 3e-5, "max": 3e-4}               # 2e-7 to 8e-6 and 2e-5 seen; gradients summed over 1e8 entries among them
