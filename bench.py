#!/usr/bin/env python3
"""Benchmark of the fused GNN sparse-operator path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload gat_c2|gat_c5|gat_c5_l2|gat_c5_train|edgeconv_c3|gmm_c4|small_ops_c2|gather_ceiling]

Default workload = benchmark configuration 2: one fused GAT layer forward+backward (dense projection, with the
scores as its last columns, and fused sparse op by libfgnn_hip.so) on a seeded R-MAT power-law graph with 232,965
nodes and ~114.6 M edges plus self loops, features [N,256], 8 heads x 32, fp32.  A step is one
layer forward + backward; inputs are resident in HBM before the timed region; graph
preprocessing (csr2csc, schedules) is reported separately.  One JSON line is printed with the
metric, the roofline record of the dominant kernel and a CPU baseline (the torch-composed DGL-style
layer of oracle/ on the host cores, on a bounded sample of the same graph).  The default run also
measures the other benchmark configurations (EdgeConv C3, GMMConv C4, GAT C5 layer 1 and the C5
training step, the small operators at C2) and appends them to the same line under "other_configs" (--no-others skips them).
gat_c5_l2 is the output layer of the C5 model alone (256 -> 1 head x 47 classes), the second half of the training step's sparse work.
Every timed call sits inside a marker range (roctx) named for the workload and the entry point, so that a kernel trace of this
file can be cut per entry point.

Roofline record: `achieved` is MEASURED bytes (rocprofv3 FETCH_SIZE + WRITE_SIZE of the entry point's
kernels, kept in profiles/traffic.json) over the live HIP-event time, `frac` its share of the 8 TB/s HBM
peak; the counters sit between L2 and the fabric, so this bounds the HBM traffic from above.  The rate of
the no-reuse gather model (one full feature row per edge and pass) is reported next to it as
`effective_gather_GBps`: it exceeds the HBM peak wherever gathered rows are served from the per-XCD L2.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

HBM_PEAK_GBPS = 8000.0      # MI355X HBM3E, published peak

TRAFFIC_FILE = os.path.join(ROOT, "profiles", "traffic.json")
CSRC_DIR = os.path.join(ROOT, "ae_mlsys_gnn_amd", "csrc")


def csrc_digest():
    """sha256 over the kernel sources: profiles/traffic.json records the digest its byte counts were measured at."""
    import glob
    import hashlib
    h = hashlib.sha256()
    for f in sorted(glob.glob(os.path.join(CSRC_DIR, "*.hip")) + glob.glob(os.path.join(CSRC_DIR, "*.h"))):
        h.update(os.path.basename(f).encode())
        with open(f, "rb") as fh:
            h.update(fh.read())
    return h.hexdigest()


def measured_traffic(workload):
    """L2<->fabric bytes per call of the entry points of `workload`, measured with rocprofv3 --pmc (FETCH_SIZE and
    WRITE_SIZE, scaled by what the same counters read for a 1 GiB copy), from profiles/traffic.json.  Returns
    (dict or None, stale): stale when the kernel sources have changed since the measurement."""
    try:
        with open(TRAFFIC_FILE) as fh:
            t = json.load(fh)
    except (OSError, ValueError):
        return None, False
    stale = t.get("csrc_sha256") != csrc_digest()
    if stale:
        print("bench.py: the kernel sources changed after profiles/traffic.json was measured (commit %s): byte counts may be stale"
              % t.get("measured_at_commit"), file=sys.stderr)
    return t.get("workloads", {}).get(workload), stale


def roofline_record(kernel, alg_bytes, ms, traffic, stale=False, note=None):
    """achieved / frac: measured L2<->fabric bytes (an upper bound on the HBM bytes) over the kernel time, against the
    HBM peak.  effective_gather_GBps: the no-reuse gather model's bytes over the same time (cache-served rows count
    in full, so it can exceed the peak).  Without a byte measurement the record falls back to the model and says so."""
    eff = alg_bytes / ms / 1e6
    rec = {"bound": "hbm", "kernel": kernel, "peak": HBM_PEAK_GBPS, "unit": "GB/s", "traffic": traffic, "alg_bytes": alg_bytes, "ms": round(ms, 4),
           "effective_gather_GBps": round(eff, 1), "effective_gather_frac": round(eff / HBM_PEAK_GBPS, 4)}
    if traffic:
        rec["achieved"] = round(traffic / ms / 1e6, 1)
        rec["frac"] = round(traffic / ms / 1e6 / HBM_PEAK_GBPS, 4)
        rec["achieved_basis"] = "measured L2<->fabric bytes (rocprofv3 FETCH_SIZE + WRITE_SIZE, profiles/traffic.json) / live HIP-event time"
        rec["limiter"] = ("L2<->fabric path; %.0f %% of the gathered bytes are served by the per-XCD L2" % (100 * (1 - traffic / alg_bytes))
                          if traffic < 0.9 * alg_bytes else "HBM")
        if stale:
            rec["traffic_stale"] = True
    else:
        rec["achieved"] = round(eff, 1)
        rec["frac"] = round(eff / HBM_PEAK_GBPS, 4)
        rec["achieved_basis"] = "algorithmic bytes (no byte-counter measurement for this kernel)"
    if note:
        rec["note"] = note
    return rec


class marker:
    """Named range around a phase of the benchmark (roctx through torch.cuda.nvtx; the counterpart of the reference's
    util/indicator.py:17-20 cudaProfilerStart/Stop brackets): `rocprofv3 --marker-trace` attributes kernels to it."""

    def __init__(self, name):
        self.name = name

    def __enter__(self):
        try:
            import torch
            torch.cuda.nvtx.range_push(self.name)
            self.ok = True
        except Exception:
            self.ok = False
        return self

    def __exit__(self, *exc):
        if self.ok:
            import torch
            torch.cuda.nvtx.range_pop()
        return False


def peak_hbm_gib():
    """Peak device memory: torch's allocator plus what the library's schedules hold outside it."""
    import torch
    from ae_mlsys_gnn_amd import _lib
    return (torch.cuda.max_memory_allocated() + _lib.schedule_device_bytes()) / 2**30


def gat_alg_bytes(n, e, h, f):
    """No-reuse gather model: every edge moves one feature row per gather pass."""
    fwd = e * (4 * h * f + 4 * h + 4) + n * (4 * h * f + 12 * h + 4)
    bwd = e * (4 * h * f + 16 * h + 4) + n * (16 * h * f + 24 * h + 4)
    return fwd, bwd


def time_calls(fn, steps, warmup, name=None):
    """Average milliseconds of fn() over `steps` calls, HIP events on torch's current stream (the
    stream every fgnn_* launch is given); the timed calls sit in a range marker called `name`."""
    import torch
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    ev = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(steps)]
    with marker(name or getattr(fn, "__name__", "timed calls")):
        for a, b in ev:
            a.record()
            fn()
            b.record()
        torch.cuda.synchronize()
    ts = [a.elapsed_time(b) for a, b in ev]
    return sum(ts) / len(ts), min(ts), sorted(ts)[len(ts) // 2]


# --permute-labels: the benchmark graphs with their node labels permuted at random (graphs.rmat_graph).  Off by default: the
# committed figures and byte counts are those of the generator's own labelling.
PERMUTE_LABELS = False


def build_gat_graph(n, e, dev, seed=0):
    import torch
    from ae_mlsys_gnn_amd import graphs
    from ae_mlsys_gnn_amd.operators import csr2csc as csc_op
    t0 = time.time()
    g = graphs.rmat_graph(n, e, seed=seed, device=dev, permute_labels=PERMUTE_LABELS)
    torch.cuda.synchronize()
    t_gen = time.time() - t0
    t0 = time.time()
    g.col_ptr, g.row_ind, g.permute = csc_op.csr2csc(g.row_ptr, g.col_ind)
    torch.cuda.synchronize()
    t_csc = time.time() - t0
    return g, t_gen, t_csc


def time_device_preprocessing(g):
    """The library's own graph pipeline on the benchmark graph: shuffled edge list -> CSR (coo2csr) ->
    CSC (csr2csc), checked against the arrays the generator produced.  Seconds, second call each."""
    import torch
    from ae_mlsys_gnn_amd.operators import csr2csc as csc_op
    dev = g.row_ptr.device
    dst = torch.repeat_interleave(torch.arange(g.n, device=dev, dtype=torch.int32), (g.row_ptr[1:] - g.row_ptr[:-1]).long())
    perm = torch.randperm(g.n_edges, device=dev)
    d2, s2 = dst[perm].contiguous(), g.col_ind[perm].contiguous()
    del dst, perm
    out = {}
    for name, fn in (("coo2csr", lambda: csc_op.coo2csr(d2, s2, g.n)), ("csr2csc", lambda: csc_op.csr2csc(g.row_ptr, g.col_ind))):
        fn()
        torch.cuda.synchronize()
        t0 = time.time()
        res = fn()
        torch.cuda.synchronize()
        out[name] = round(time.time() - t0, 4)
        if name == "coo2csr":
            out["coo2csr_matches"] = bool(torch.equal(res[0], g.row_ptr) and torch.equal(res[1], g.col_ind))
    return out


def sample_rows_subgraph(g, target_edges):
    """(row_ptr, col_ind, edges, rows) of the sub-graph formed by a seeded random sample of destination rows of `g` holding
    about `target_edges` edges (all other rows empty; every source node kept), on the host."""
    import torch
    rp = g.row_ptr.cpu().long()
    deg = rp[1:] - rp[:-1]
    order = torch.randperm(g.n, generator=torch.Generator().manual_seed(12345))
    r = int(torch.searchsorted(torch.cumsum(deg[order], 0), torch.tensor([target_edges])).item()) + 1
    r = max(1, min(r, g.n))
    rows = torch.sort(order[:r]).values
    keep = torch.zeros(g.n, dtype=torch.long)
    keep[rows] = deg[rows]
    rp_s = torch.cat([torch.zeros(1, dtype=torch.long), torch.cumsum(keep, 0)]).to(torch.int32)
    e_s = int(rp_s[-1])
    seg = torch.repeat_interleave(torch.arange(r), deg[rows])
    pos = rp[rows][seg] + (torch.arange(e_s) - (torch.cumsum(deg[rows], 0) - deg[rows])[seg])
    return rp_s, g.col_ind.cpu()[pos], e_s, r


def cpu_baseline_small_ops(g, h, f, target_edges):
    """The stand-alone operators on the host cores (oracle: u_add_v, LeakyReLU, edge softmax, multi-head SpMM, forward and
    backward by autograd) on a sampled sub-graph, scaled to the full edge count: ms for the whole chain."""
    import torch
    from oracle import fgnn_oracle as orc
    cores = os.cpu_count() or 1
    torch.set_num_threads(cores)
    rp_s, ci_s, e_s, r = sample_rows_subgraph(g, target_edges)
    gen = torch.Generator().manual_seed(3)
    ar = torch.randn(g.n, h, generator=gen).requires_grad_(True)
    ac = torch.randn(g.n, h, generator=gen).requires_grad_(True)
    x = torch.randn(g.n, h, f, generator=gen).requires_grad_(True)
    go = torch.randn(g.n, h, f, generator=gen)

    def step():
        e = torch.nn.functional.leaky_relu(orc.u_add_v(rp_s, ci_s, ar, ac), 0.2)
        orc.mhspmm(rp_s, ci_s, orc.edge_softmax(rp_s, e), x).backward(go)
        ar.grad = None; ac.grad = None; x.grad = None
    step()
    ts, t_all = [], time.time()
    while len(ts) < 3 or (time.time() - t_all < 6.0 and len(ts) < 10):
        t0 = time.time()
        step()
        ts.append((time.time() - t0) * 1e3)
    ms = sorted(ts)[len(ts) // 2]
    return {"value": round(ms * g.n_edges / e_s, 1), "unit": "ms for u_add_v + LeakyReLU + edge softmax + mhspmm, forward and backward", "cores": cores,
            "kind": "port", "sample": "oracle operators (torch CPU, %d threads) on a seeded random sample of %d destination rows = %d edges of the same "
            "graph: median %.1f ms over %d iters, scaled by E/E_sample = %.1f" % (cores, r, e_s, ms, len(ts), g.n_edges / e_s)}


def cpu_baseline_gat(g, x_feat, layer, slope, target_edges, go):
    """The DGL-composed GAT layer (oracle.gat_layer_dgl: u_add_v, LeakyReLU, edge softmax,
    u_mul_e + sum in plain torch) forward+backward on the host cores, on the sub-graph formed by a
    seeded random sample of destination rows of the benchmark graph holding about `target_edges` edges
    (all other rows empty; every source node kept); scaled to the full edge count."""
    import torch
    from oracle import fgnn_oracle as orc
    cores = os.cpu_count() or 1
    torch.set_num_threads(cores)
    rp_s, ci_s, e_s, r = sample_rows_subgraph(g, target_edges)
    feat = x_feat.detach().cpu()
    w_t = layer.W.detach().cpu().t().contiguous().requires_grad_(True)
    # weight mapping to GATConv_dgl: attn_l(dgl) = attn_r(ours), attn_r(dgl) = attn_l(ours)
    al = layer.attn_r.detach().cpu().clone().requires_grad_(True)
    ar = layer.attn_l.detach().cpu().clone().requires_grad_(True)
    go_c = go.detach().cpu()

    def step():
        out = orc.gat_layer_dgl(w_t, al, ar, rp_s, ci_s, slope, feat)
        out.backward(go_c)
        w_t.grad = None; al.grad = None; ar.grad = None

    step()
    ts = []
    t_all = time.time()
    while len(ts) < 3 or (time.time() - t_all < 10.0 and len(ts) < 20):
        t0 = time.time()
        step()
        ts.append((time.time() - t0) * 1e3)
    ms = sorted(ts)[len(ts) // 2]
    return ms, e_s, r, cores, len(ts)


def cpu_baseline_c1():
    """benchmark configuration 1 at its real size on the host: the DGL-composed GAT layer forward+backward,
    N=4096, 32,768 uniform random edges + self loops, X [4096,64], 4 heads x 16, slope 0.2, loss = sum."""
    import torch
    from ae_mlsys_gnn_amd import graphs
    from oracle import fgnn_oracle as orc
    cores = os.cpu_count() or 1
    torch.set_num_threads(cores)
    torch.manual_seed(0)
    g = graphs.uniform_graph(4096, 32768, seed=0)
    x = torch.randn(4096, 64)
    w = torch.nn.init.xavier_normal_(torch.empty(64, 64)).requires_grad_(True)
    al = (torch.randn(1, 4, 16) * 0.1).requires_grad_(True)
    ar = (torch.randn(1, 4, 16) * 0.1).requires_grad_(True)

    def step():
        orc.gat_layer_dgl(w, al, ar, g.row_ptr, g.col_ind, 0.2, x).sum().backward()
        w.grad = None; al.grad = None; ar.grad = None

    for _ in range(5):
        step()
    ts = []
    for _ in range(20):
        t0 = time.time()
        step()
        ts.append((time.time() - t0) * 1e3)
    return {"value": round(sorted(ts)[len(ts) // 2], 3), "min": round(min(ts), 3), "unit": "ms/iter", "cores": cores, "kind": "port",
            "sample": "config C1 at full size (N=4096, E=%d), DGL-composed GAT layer in torch CPU, 5 warm-up + 20 timed, median" % g.n_edges}


def run_gat(args, n, e_target, in_feats, heads, out_feats, workload):
    import torch
    from ae_mlsys_gnn_amd import _lib
    from ae_mlsys_gnn_amd.layers import GATConv
    from ae_mlsys_gnn_amd.operators.fused_gat import gat_native
    dev = torch.device("cuda:0")
    torch.manual_seed(0)
    g, t_gen, t_csc = build_gat_graph(n, e_target, dev)
    e = g.n_edges
    t0 = time.time()
    s_csr = _lib.schedule_for(g.row_ptr, idx_tensor=g.col_ind, need_positions=False)
    s_csc = _lib.schedule_for(g.col_ptr, idx_tensor=g.row_ind, need_positions=False)
    torch.cuda.synchronize()
    t_sched = time.time() - t0
    slope = 0.2
    layer = GATConv(in_feats, out_feats, heads, slope).to(dev)
    with torch.no_grad():          # config: attn_l / attn_r ~ N(0, 0.1)
        layer.attn_l.normal_(0, 0.1)
        layer.attn_r.normal_(0, 0.1)
    x = torch.randn(n, in_feats, device=dev)
    go = torch.randn(n, heads, out_feats, device=dev)

    def step():
        out = layer(g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, x)
        out.backward(go)
        for p in layer.parameters():
            p.grad = None

    # timed region: exactly K steps between two synchronisations
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    with marker(workload + ": layer forward + backward, timed steps"):
        for _ in range(args.steps):
            step()
        torch.cuda.synchronize()
    ms_step = (time.perf_counter() - t0) * 1e3 / args.steps

    # dominant kernels alone, through the C ABI, HIP events on the launch stream
    with torch.no_grad():
        h = torch.matmul(x, layer.W).view(-1, heads, out_feats).contiguous()
        a_row = (layer.attn_l * h).sum(-1).contiguous()
        a_col = (layer.attn_r * h).sum(-1).contiguous()
    go_k, f_k = go, out_feats
    if out_feats % 4:          # an output layer: the layer zero-pads its rows to a multiple of four floats (128-bit lanes); so does this
        f_k = out_feats + (-out_feats) % 4
        h = torch.nn.functional.pad(h, (0, f_k - out_feats)).contiguous()
        go_k = torch.nn.functional.pad(go, (0, f_k - out_feats)).contiguous()
    fwd_out = gat_native.gat_forward(a_row, a_col, g.row_ptr, g.col_ind, slope, h)
    ms_fwd, ms_fwd_min, _ = time_calls(lambda: gat_native.gat_forward(a_row, a_col, g.row_ptr, g.col_ind, slope, h), args.steps, 2, workload + ": fgnn_gat_forward")
    o = fwd_out
    ms_bwd, ms_bwd_min, _ = time_calls(
        lambda: gat_native.gat_backward(slope, g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, o[1], o[2], h, a_row, a_col, go_k,
                                        out_feat=o[0], out2=o[3], cc=o[4]), args.steps, 2, workload + ": fgnn_gat_backward")
    b_fwd, b_bwd = gat_alg_bytes(n, e, heads, f_k)
    traffic, stale = measured_traffic(workload)
    peak_mem = peak_hbm_gib()
    # stash variant as the autograd function runs it: the attention [E,H] written after the forward in the entry order of
    # the backward pass (signed: the sign bit says whether the pre-activation was positive) and streamed by the backward
    own = gat_native.gat_stash_own_order(slope, g.col_ptr, g.row_ind, o[1], o[2], a_row, a_col)
    ms_sw, _, _ = time_calls(lambda: gat_native.gat_stash_own_order(slope, g.col_ptr, g.row_ind, o[1], o[2], a_row, a_col), max(3, args.steps // 4), 1)
    ms_sf = ms_fwd + ms_sw
    ms_sb, _, _ = time_calls(
        lambda: gat_native.gat_backward(slope, g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, o[1], o[2], h, a_row, a_col, go_k,
                                        out_feat=o[0], out2=o[3], cc=o[4], e_soft=own, e_soft_order="own"),
        max(3, args.steps // 4), 1)
    stash_bytes = e * heads * 4
    del own, o, fwd_out
    x = x.cpu()          # the pipelines below start from the projected features h; the host baseline takes the input from the host
    # the reference's fuse-scatter variant with its own data flow (scatter kernel -> e_softmax [E,H] -> multi-head SpMM; backward
    # by permuted SpMM, SDDMM, gather-row kernel and column sums), and the same layer composed from the stand-alone operators
    from ae_mlsys_gnn_amd.operators.fused_gat import fused_gat_fusescatter_pipeline, fused_gat_operator_pipeline
    pipes = {}
    for pname, pfn in (("fusescatter", fused_gat_fusescatter_pipeline), ("operators", fused_gat_operator_pipeline)):
        hp, arp, acp = (t.detach().clone().requires_grad_(True) for t in (h, a_row, a_col))

        def pipeline_step():
            pfn(arp, acp, g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, slope, hp, g.permute).backward(go_k)
            hp.grad = None; arp.grad = None; acp.grad = None
        _lib.clear_schedule_cache()          # each variant is charged its own work lists and plans only
        torch.cuda.empty_cache()
        torch.cuda.reset_peak_memory_stats()
        ms_p, _, _ = time_calls(pipeline_step, max(3, args.steps // 4), 1, workload + ": pipeline " + pname)
        pipes[pname] = (ms_p, peak_hbm_gib())
        del hp, arp, acp
    ms_pipe, pipe_peak = pipes["fusescatter"]
    prep = time_device_preprocessing(g)

    if args.no_cpu_baseline:
        cpu_ms, cpu_e, cpu_rows, cores, cpu_iters = float("nan"), e, 0, 0, 0
    else:
        cpu_ms, cpu_e, cpu_rows, cores, cpu_iters = cpu_baseline_gat(g, x, layer, slope, args.cpu_sample_edges, go)
    c1 = None if (args.no_cpu_baseline or workload != "gat_c2") else cpu_baseline_c1()
    rec = {
        "metric": "GAT layer fwd+bwd ms/iter + achieved HBM GB/s (% of peak), 1 MI355X",
        "value": round(ms_step, 4), "unit": "ms/iter", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(ms_step, 4), "higher_is_better": False, "scaling": "weak", "vs_baseline": None,
        "dtype": "f32", "data": "synthetic",
        "config": {"workload": workload, "graph": "R-MAT a=0.57 b=0.19 c=0.19 d=0.05 seed 0, unique edges + self loops" + (", node labels permuted" if PERMUTE_LABELS else ""),
                   "nodes": n, "edges": e, "in_feats": in_feats, "heads": heads, "out_feats": out_feats,
                   "negative_slope": slope, "step": "GATConv forward + backward (fp32 projection with the scores as its last columns + fused sparse op)"},
        "roofline": roofline_record("gat_fwd_kernel (+gat_fwd_merge_kernel)", b_fwd, ms_fwd, (traffic or {}).get("fwd"), stale),
        "roofline_bwd": roofline_record("gat_bwd_node_kernel + gat_bwd_kernel (+gat_bwd_merge_kernel)", b_bwd, ms_bwd,
                                        (traffic or {}).get("bwd"), stale),
        "stash_variant": {"fwd_ms": round(ms_sf, 4), "stash_writer_ms": round(ms_sw, 4), "bwd_ms": round(ms_sb, 4),
                          "stashed_GiB": round(stash_bytes / 2**30, 3),
                          "roofline_bwd": roofline_record("gat_bwd_node_kernel + gat_bwd_kernel<own-order stash> (+merge)", b_bwd + stash_bytes, ms_sb,
                                                          (traffic or {}).get("stash_bwd"), stale)},
        "fusescatter_pipeline": {"fwd_bwd_ms": round(ms_pipe, 4), "peak_hbm_GiB": round(pipe_peak, 3),
                                 "what": "the reference's fuse-scatter variant in its own data flow: scatter kernel -> e_softmax [E,H] -> mhspmm; "
                                         "backward by permuted mhspmm, mhsddmm, gather-row kernel, column sums",
                                 "composed_from_standalone_operators": {"fwd_bwd_ms": round(pipes["operators"][0], 4),
                                                                        "peak_hbm_GiB": round(pipes["operators"][1], 3)}},
        "sparse_fwd_bwd": {"ms": round(ms_fwd + ms_bwd, 4), "alg_bytes": b_fwd + b_bwd,
                           "effective_gather_GBps": round((b_fwd + b_bwd) / (ms_fwd + ms_bwd) / 1e6, 1),
                           "measured_GBps": (round((traffic["fwd"] + traffic["bwd"]) / (ms_fwd + ms_bwd) / 1e6, 1)
                                             if traffic and "fwd" in traffic and "bwd" in traffic else None)},
        "cpu_baseline": None if args.no_cpu_baseline else {
            "value": round(cpu_ms * e / cpu_e, 1), "unit": "ms/iter", "cores": cores, "kind": "port",
            "sample": "DGL-composed GAT layer (torch CPU, %d threads) fwd+bwd on a seeded random sample of %d destination rows = %d edges of the "
                      "same graph: median %.1f ms over %d iters, scaled by E/E_sample = %.1f" % (cores, cpu_rows, cpu_e, cpu_ms, cpu_iters, e / cpu_e)},
        "cpu_baseline_c1": c1,
        "preprocess_s": {"graph_gen": round(t_gen, 3), "csr2csc_first_call": round(t_csc, 4), "schedules": round(t_sched, 4), **prep},
        "schedule": {"xcd_aware": s_csr.idx_tensor is not None, "csr_items": s_csr.n_items, "csr_partials": s_csr.n_partials,
                     "csc_items": s_csc.n_items, "csc_partials": s_csc.n_partials,
                     "device_GiB": round((s_csr.device_bytes() + s_csc.device_bytes()) / 2**30, 3)},
        "peak_hbm_GiB": round(peak_mem, 3),
    }
    return rec


def run_edgeconv(args):
    import torch
    from ae_mlsys_gnn_amd import graphs
    from ae_mlsys_gnn_amd.operators.fused_edgeconv import edgeconv_native
    from ae_mlsys_gnn_amd.operators.knn import knn_graph
    from oracle import fgnn_oracle as orc
    dev = torch.device("cuda:0")
    torch.manual_seed(0)
    bsz, npts, k, f = 32, 1024, 20, 64
    pts = (torch.rand(bsz, npts, 3, device=dev) * 2 - 1)
    src = graphs.knn_graph(pts, k)
    n = bsz * npts
    theta = torch.nn.Linear(3, f, bias=False).to(dev)
    phi = torch.nn.Linear(3, f, bias=False).to(dev)
    xin = pts.reshape(-1, 3)
    with torch.no_grad():
        h_src = theta(xin).contiguous()
        h_dst = (phi(xin) - h_src).contiguous()
    go = torch.randn(n, f, device=dev)
    out, arg = edgeconv_native.edgeconv_forward(k, src, h_src, h_dst)
    ms_f, _, _ = time_calls(lambda: edgeconv_native.edgeconv_forward(k, src, h_src, h_dst), args.steps, args.warmup)
    ms_b_plain, _, _ = time_calls(lambda: edgeconv_native.edgeconv_backward(go, arg, n), args.steps, args.warmup)
    # the graph is a kNN graph of clouds of npts points: the backward may accumulate per cloud in LDS
    ms_b, _, _ = time_calls(lambda: edgeconv_native.edgeconv_backward(go, arg, n, block=npts), args.steps, args.warmup)
    # the step is launch-bound: captured into a HIP graph the host-side gaps disappear
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        edgeconv_native.edgeconv_backward(go, edgeconv_native.edgeconv_forward(k, src, h_src, h_dst)[1], n, block=npts)
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g_out, g_arg = edgeconv_native.edgeconv_forward(k, src, h_src, h_dst)
        g_gs = edgeconv_native.edgeconv_backward(go, g_arg, n, block=npts)
    ms_graph, _, _ = time_calls(graph.replay, args.steps, args.warmup)
    graph_ok = bool(torch.equal(g_out, out) and torch.equal(g_arg, arg))
    knn_graph(pts, k)
    ms_knn, _, _ = time_calls(lambda: knn_graph(pts, k), args.steps, args.warmup)
    e = n * k
    traffic, stale = measured_traffic("edgeconv_c3")
    b_f = e * (4 * f + 4) + n * f * 12
    b_b = n * f * 20
    # CPU baseline: EdgeConv_reorg composed math on the host, full size (it is small)
    cores = os.cpu_count() or 1
    torch.set_num_threads(cores)
    hs_c, hd_c, src_c = h_src.cpu().requires_grad_(True), h_dst.cpu().requires_grad_(True), src.cpu()
    go_c = go.cpu()
    ts = []
    for _ in range(5):
        t0 = time.time()
        o = orc.edgeconv_forward_autograd(k, src_c, hs_c, hd_c)
        o.backward(go_c)
        hs_c.grad = None; hd_c.grad = None
        ts.append((time.time() - t0) * 1e3)
    ms = ms_f + ms_b
    return {
        "metric": "fused EdgeConv fwd+bwd us/iter + achieved GB/s, 1 MI355X", "value": round(ms * 1e3, 2), "unit": "us/iter", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms, 5), "higher_is_better": False, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": "edgeconv_c3", "clouds": bsz, "points": npts, "k": k, "F": f, "edges": e},
        "hip_graph_replay": {"fwd_bwd_us": round(ms_graph * 1e3, 2), "matches_eager": graph_ok},
        "knn_graph_ms": round(ms_knn, 3),
        "roofline": roofline_record("edgeconv_fwd_kernel", b_f, ms_f, (traffic or {}).get("fwd"), stale,
                                    note="237 MB of algorithmic bytes: launch-latency bound, not bandwidth bound"),
        "roofline_bwd": roofline_record("edgeconv_bwd_blocked_kernel (+ overflow kernel)", b_b, ms_b, (traffic or {}).get("bwd_blocked"), stale),
        "backward_plain_scatter_us": round(ms_b_plain * 1e3, 2),
        "cpu_baseline": {"value": round(sorted(ts)[len(ts) // 2] * 1e3, 1), "unit": "us/iter", "cores": cores, "kind": "port",
                         "sample": "EdgeConv_reorg composed math (torch CPU gather + max over k) fwd+bwd at full size, median of 5"},
    }


def run_gmm(args):
    import torch
    from ae_mlsys_gnn_amd import _lib
    from ae_mlsys_gnn_amd.operators.fused_gmmconv import gmm_native
    from oracle import fgnn_oracle as orc
    dev = torch.device("cuda:0")
    torch.manual_seed(0)
    n, e_t, kk, dim, f = 169343, 2_300_000, 3, 2, 64
    g, t_gen, t_csc = build_gat_graph(n, e_t, dev, seed=1)
    e = g.n_edges
    deg = (g.row_ptr[1:] - g.row_ptr[:-1]).float()
    dst = torch.repeat_interleave(torch.arange(n, device=dev), (g.row_ptr[1:] - g.row_ptr[:-1]).long())
    src = g.col_ind.long()
    pseudo = torch.stack([deg[src].rsqrt(), deg[dst].rsqrt()], 1).contiguous()      # CSR position order
    x = torch.randn(n, kk, f, device=dev)
    mu = torch.rand(kk, dim, device=dev)
    isg = torch.ones(kk, dim, device=dev)
    go = torch.randn(n, kk, f, device=dev)
    _lib.schedule_for(g.row_ptr); _lib.schedule_for(g.col_ptr)
    ms_f, _, _ = time_calls(lambda: gmm_native.gmmconv(g.row_ptr, g.col_ind, x, pseudo, mu, isg), args.steps, args.warmup)
    ms_b, _, _ = time_calls(lambda: gmm_native.gmmconv_backward(g.col_ptr, g.row_ind, g.permute, x, pseudo, mu, isg, go), args.steps, args.warmup)
    # the layer's form: sum over the K kernels fused into the operator ([N,F] out, [N,F] gradient rows gathered)
    go_s = go[:, 0, :].contiguous()
    ms_fs, _, _ = time_calls(lambda: gmm_native.gmmconv(g.row_ptr, g.col_ind, x, pseudo, mu, isg, sum_kernels=True), args.steps, args.warmup)
    ms_bs, _, _ = time_calls(lambda: gmm_native.gmmconv_backward(g.col_ptr, g.row_ind, g.permute, x, pseudo, mu, isg, go_s, sum_kernels=True),
                             args.steps, args.warmup)
    traffic, stale = measured_traffic("gmm_c4")
    b_f = e * (4 * kk * f + 4 * dim + 4) + n * (4 * kk * f + 4)
    b_b = e * (4 * kk * f + 8 * dim + 12) + n * (8 * kk * f + 4)
    cores = os.cpu_count() or 1
    torch.set_num_threads(cores)
    leaves = [t.cpu().requires_grad_(True) for t in (x, pseudo, mu, isg)]
    rp_c, ci_c, go_c = g.row_ptr.cpu(), g.col_ind.cpu(), go.cpu()
    ts = []
    for _ in range(3):
        t0 = time.time()
        orc.gmm_forward(rp_c, ci_c, *leaves).backward(go_c)
        for t in leaves:
            t.grad = None
        ts.append((time.time() - t0) * 1e3)
    ms = ms_f + ms_b
    return {
        "metric": "fused GMMConv fwd+bwd ms/iter + achieved GB/s, 1 MI355X", "value": round(ms, 4), "unit": "ms/iter", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms, 4), "higher_is_better": False, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": "gmm_c4", "nodes": n, "edges": e, "K": kk, "dim": dim, "F": f},
        "roofline": roofline_record("spmm_kernel<WGauss>", b_f, ms_f, (traffic or {}).get("fwd"), stale),
        "roofline_bwd": roofline_record("gmm_bwd_kernel + gauss_grad_small_kernel + column sums", b_b, ms_b, (traffic or {}).get("bwd"), stale),
        "fused_sum_over_kernels": {"fwd_ms": round(ms_fs, 4), "bwd_ms": round(ms_bs, 4)},
        "cpu_baseline": {"value": round(sorted(ts)[1], 1), "unit": "ms/iter", "cores": cores, "kind": "port",
                         "sample": "GMMConv_dgl composed math (torch CPU) fwd+bwd at full size, median of 3"},
    }


def run_gat_train(args):
    """benchmark configuration 5: full 2-layer GAT training step (forward, cross-entropy over all nodes,
    backward, Adam) with the model of the reference's script/train/train_gatconv_our.py:33-53
    (GATConv(100, 32, 8) -> flatten -> GATConv(256, 47, 1) -> mean over heads; no activation in
    between), recompute variant against stash variant; reports ms/step and peak HBM of both."""
    import torch
    from torch import nn
    from ae_mlsys_gnn_amd import _lib
    from ae_mlsys_gnn_amd.layers import GATConv, GATConv_stash
    from ae_mlsys_gnn_amd.train.common import cross_entropy, head_mean
    dev = torch.device("cuda:0")
    n, e_t, in_dim, hidden, heads, classes = 2449029, 61_900_000, 100, 32, 8, 47
    g, t_gen, t_csc = build_gat_graph(n, e_t, dev)
    e = g.n_edges
    _lib.schedule_for(g.row_ptr); _lib.schedule_for(g.col_ptr)
    torch.manual_seed(0)
    x = torch.randn(n, in_dim, device=dev)
    labels = torch.randint(0, classes, (n,), device=dev)

    class GAT(nn.Module):
        def __init__(self, conv):
            super().__init__()
            self.l1 = conv(in_dim, hidden, heads, 0.2)
            self.l2 = conv(hidden * heads, classes, 1, 0.2)

        def forward(self, extra):
            h = self.l1(g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, x, extra).flatten(1)
            # the logits keep the output layer's zero column (47 -> 48): the loss takes the class count instead of a cropped view
            return head_mean(self.l2(g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, h, extra, keep_padding=True))

    res = {}
    for name, conv, extra in (("recompute", GATConv, True), ("stash", GATConv_stash, g.permute)):
        torch.manual_seed(1)
        model = GAT(conv).to(dev)
        opt = torch.optim.Adam(model.parameters(), lr=5e-3, weight_decay=5e-4)
        loss_fn = cross_entropy

        def step():
            logits = model(extra)
            loss = loss_fn(logits, labels, classes)
            opt.zero_grad()
            loss.backward()
            opt.step()
            return loss

        torch.cuda.empty_cache()
        torch.cuda.reset_peak_memory_stats()
        base = torch.cuda.memory_allocated()
        for _ in range(args.warmup):
            step()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        with marker("gat_c5_train: " + name + ", timed steps"):
            for _ in range(args.steps):
                loss = step()
            torch.cuda.synchronize()
        ms = (time.perf_counter() - t0) * 1e3 / args.steps
        res[name] = {"ms_per_step": round(ms, 3), "peak_hbm_GiB": round(peak_hbm_gib(), 3),
                     "of_which_schedules_GiB": round(_lib.schedule_device_bytes() / 2**30, 3),
                     "resident_before_GiB": round(base / 2**30, 3), "final_loss": round(float(loss.detach()), 5)}
        del model, opt
        if name == "recompute":
            # the same step captured once into a HIP graph and replayed (same number of optimizer steps from the same start):
            # what the launch gaps between the step's ~100 kernels are worth at this size
            from ae_mlsys_gnn_amd.train.common import capture_step
            torch.manual_seed(1)
            model = GAT(conv).to(dev)
            opt = torch.optim.Adam(model.parameters(), lr=5e-3, weight_decay=5e-4, capturable=True)
            replay = capture_step(step, dev, warmup=args.warmup)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            with marker("gat_c5_train: recompute, HIP-graph replays"):
                for _ in range(args.steps):
                    loss = replay()
                torch.cuda.synchronize()
            res[name]["hip_graph_ms_per_step"] = round((time.perf_counter() - t0) * 1e3 / args.steps, 3)
            res[name]["hip_graph_final_loss"] = round(float(loss.detach()), 5)
            del model, opt, replay
    b1 = gat_alg_bytes(n, e, heads, hidden)
    b2 = gat_alg_bytes(n, e, 1, classes)
    alg = sum(b1) + sum(b2)
    ms = res["recompute"]["ms_per_step"]
    # measured bytes of the step's sparse entry points: both layers, forward and backward
    t1, stale1 = measured_traffic("gat_c5_layer1")
    t2, stale2 = measured_traffic("gat_c5_layer2")
    traffic = (t1["fwd"] + t1["bwd"] + t2["fwd"] + t2["bwd"]) if (t1 and t2 and all(k in t for t in (t1, t2) for k in ("fwd", "bwd"))) else None
    return {
        "metric": "2-layer GAT training step ms/step + peak HBM, recompute vs stash, 1 MI355X", "value": ms, "unit": "ms/step",
        "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": ms, "higher_is_better": False, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": "gat_c5_train", "nodes": n, "edges": e, "in_feats": in_dim, "hidden": "8x32", "classes": classes,
                   "optimizer": "Adam(lr=5e-3, weight_decay=5e-4)", "loss": "mean cross-entropy over all nodes (fused row pass: logsumexp - true-class logit)"},
        "variants": res,
        "roofline": roofline_record("whole step (sparse ops of both layers; dense GEMMs, loss and Adam included in the time)", alg, ms, traffic,
                                    stale1 or stale2, note="traffic = measured bytes of fgnn_gat_forward + fgnn_gat_backward of both layers "
                                    "(gat_c5_layer1 + gat_c5_layer2 of profiles/traffic.json); the GEMMs, the loss and Adam add time but are not in the bytes"),
        "cpu_baseline": None,
    }


def run_gather_ceiling(args):
    """What a bare feature-row gather reaches on this part, with the library's own unweighted SpMM (fgnn_mhspmm
    without weights: one 1 KiB row gathered and added per edge, nothing else per edge): on the C2 graph as it is
    (skewed sources, XCD-aware work list) and with every source replaced by a uniform random node (no reuse to
    speak of: the rate of the L2<->fabric path itself), likewise at the C5 size (features far larger than the caches)."""
    import torch
    from ae_mlsys_gnn_amd import _lib, graphs
    from ae_mlsys_gnn_amd.operators import mhspmm as mh
    dev = torch.device("cuda:0")
    h, f = 8, 32
    out = {}
    for name, n, e_t in (("c2_graph", 232965, 114_600_000), ("c5_graph", 2449029, 61_900_000)):
        g = graphs.rmat_graph(n, e_t, seed=0, device=dev, permute_labels=PERMUTE_LABELS)
        e = g.n_edges
        x = torch.randn(n, h, f, device=dev)
        alg = e * (4 * h * f + 4) + n * 4 * h * f
        ms_skew, _, _ = time_calls(lambda: mh.mhspmm(g.row_ptr, g.col_ind, None, x), args.steps, 2)
        ci = torch.randint(0, n, (e,), device=dev, dtype=torch.int32)
        ms_unif, _, _ = time_calls(lambda: mh.mhspmm(g.row_ptr, ci, None, x), args.steps, 2)
        out[name] = {"nodes": n, "edges": e, "row_bytes": 4 * h * f, "alg_bytes": alg,
                     "own_sources": {"ms": round(ms_skew, 4), "effective_gather_GBps": round(alg / ms_skew / 1e6, 1)},
                     "uniform_random_sources": {"ms": round(ms_unif, 4), "effective_gather_GBps": round(alg / ms_unif / 1e6, 1),
                                                "frac_of_hbm_peak": round(alg / ms_unif / 1e6 / HBM_PEAK_GBPS, 4)}}
        del g, x, ci
        _lib.clear_schedule_cache()
        torch.cuda.empty_cache()
    # what plain streaming kernels of the installed libraries reach on this part (no gather at all): the practical
    # ceiling next to the published 8 TB/s
    stream = {}
    for mib in (256, 4096):
        nel = mib * 1024 * 1024 // 4
        a = torch.randn(nel, device=dev)
        b = torch.empty_like(a)
        for name, nbytes, fn in (("copy", 8 * nel, lambda: b.copy_(a)), ("scale (read + write)", 8 * nel, lambda: torch.mul(a, 2.0, out=b)),
                                 ("fill", 4 * nel, lambda: b.zero_()), ("sum (read only)", 4 * nel, lambda: a.sum())):
            t, _, _ = time_calls(fn, args.steps, 3)
            stream["%s, %d MiB arrays" % (name, mib)] = {"ms": round(t, 4), "GBps": round(nbytes / t / 1e6, 1),
                                                         "frac_of_hbm_peak": round(nbytes / t / 1e6 / HBM_PEAK_GBPS, 4)}
        del a, b
        torch.cuda.empty_cache()
    out["library_streaming_kernels"] = stream
    ms = out["c2_graph"]["uniform_random_sources"]["ms"]
    return {"metric": "bare 1 KiB feature-row gather (unweighted SpMM) ms + GB/s, 1 MI355X", "value": ms, "unit": "ms/iter", "n_gpus": 1,
            "steps": args.steps, "warmup": 2, "ms_per_step": ms, "higher_is_better": False, "scaling": "weak", "vs_baseline": None,
            "dtype": "f32", "data": "synthetic", "config": {"workload": "gather_ceiling", "heads": h, "out_feats": f}, "graphs": out,
            "roofline": roofline_record("spmm_kernel (unweighted), uniform random sources on the C2 degree sequence",
                                        out["c2_graph"]["alg_bytes"], ms, None), "cpu_baseline": None}


def run_small_ops(args):
    """The per-edge operators of the reference's operators/ package on the C2 graph, each timed alone: u_add_v, edge
    softmax, multi-head SpMM / SDDMM, the permuted row gather, csr2csc.  `bytes` is what one call must move when
    nothing is reused: every array read or written once, gathered feature rows once per entry."""
    import torch
    from ae_mlsys_gnn_amd import _lib
    from ae_mlsys_gnn_amd.operators import csr2csc as csc_op
    from ae_mlsys_gnn_amd.operators import fused_gat as fg
    from ae_mlsys_gnn_amd.operators import mhspmm as mh
    from ae_mlsys_gnn_amd.operators.edge_softmax import edge_softmax_native
    from ae_mlsys_gnn_amd.operators.u_add_v import u_add_v_native
    dev = torch.device("cuda:0")
    n, h, f = 232965, 8, 32
    g, _, _ = build_gat_graph(n, 114_600_000, dev)
    e = g.n_edges
    torch.manual_seed(0)
    x = torch.randn(n, h, f, device=dev)
    go = torch.randn(n, h, f, device=dev)
    ar = torch.randn(n, h, device=dev)
    ac = torch.randn(n, h, device=dev)
    ee = u_add_v_native.u_add_v_forward(g.row_ptr, g.col_ind, ar, ac)
    sm = edge_softmax_native.edge_softmax(g.row_ptr, ee)
    eh, nh, row = 4 * e * h, 4 * n * h, 4 * h * f
    ops = (
        ("u_add_v", "fgnn_u_add_v", eh + 4 * e + 2 * nh, lambda: u_add_v_native.u_add_v_forward(g.row_ptr, g.col_ind, ar, ac)),
        ("u_add_v_backward", "fgnn_u_add_v_backward_planned (row sums + column sums under a plan, no atomics)", 2 * eh + 2 * nh,
         lambda: u_add_v_native.u_add_v_backward(g.row_ptr, g.col_ind, ee)),
        ("u_add_v_backward_atomics", "fgnn_u_add_v_backward", eh + 4 * e + 2 * nh,
         lambda: u_add_v_native.u_add_v_backward(g.row_ptr, g.col_ind, ee, atomics=True)),
        ("edge_softmax", "fgnn_edge_softmax", 2 * eh, lambda: edge_softmax_native.edge_softmax(g.row_ptr, ee)),
        ("edge_softmax_backward", "fgnn_edge_softmax_backward", 3 * eh, lambda: edge_softmax_native.edge_softmax_backward(g.row_ptr, sm, ee)),
        ("mhspmm", "fgnn_mhspmm", e * (row + 4 + 4 * h) + n * row, lambda: mh.mhspmm(g.row_ptr, g.col_ind, sm, x)),
        ("mhspmm_transposed", "fgnn_mhspmm (CSC walk, weights through permute)", e * (row + 8 + 4 * h) + n * row,
         lambda: mh.mhspmm(g.col_ptr, g.row_ind, sm, go, pos_map=g.permute)),
        ("mhsddmm", "fgnn_mhsddmm", e * (row + 4 + 4 * h) + n * row, lambda: mh.mhsddmm(g.row_ptr, g.col_ind, go, x)),
        ("mhtranspose", "fgnn_gather_rows", 2 * eh + 4 * e, lambda: mh.mhtranspose(g.permute, sm)),
        ("gat_scatter", "fgnn_gat_scatter", eh + 4 * e + 2 * nh, lambda: fg.gat_native.gat_scatter(ar, ac, g.row_ptr, g.col_ind, 0.2)),
        ("gat_gather_row", "fgnn_gat_gather_row", 3 * eh, lambda: fg.gat_native.gat_gather_row(0.2, g.row_ptr, g.col_ind, ar, ac, sm, ee)),
        ("csr2csc", "fgnn_csr2csc", 0, lambda: csc_op.csr2csc(g.row_ptr, g.col_ind)),
    )
    out = {}
    traffic, stale = measured_traffic("small_ops_c2")
    traffic = traffic or {}
    for name, entry, nbytes, fn in ops:
        ms, _, _ = time_calls(fn, min(args.steps, 10), 2, "small_ops_c2: " + name)
        out[name] = {"entry_point": entry, "ms": round(ms, 3)}
        if name in traffic:          # L2<->fabric bytes by the byte counters: above `bytes` where rows are fetched as whole 128-byte lines or read twice
            out[name].update({"traffic": traffic[name], "traffic_GBps": round(traffic[name] / ms / 1e6, 1),
                              "traffic_frac_of_hbm_peak": round(traffic[name] / ms / 1e6 / HBM_PEAK_GBPS, 4)})
            if stale:
                out[name]["traffic_stale"] = True
        if nbytes and name.startswith("mh") and name != "mhtranspose":
            # feature rows gathered once per entry by the model, mostly served by the L2s: a rate, not a share of the HBM peak
            out[name].update({"no_reuse_model_bytes": nbytes, "effective_gather_GBps": round(nbytes / ms / 1e6, 1)})
        elif nbytes:
            out[name].update({"bytes": nbytes, "GBps": round(nbytes / ms / 1e6, 1), "frac_of_hbm_peak": round(nbytes / ms / 1e6 / HBM_PEAK_GBPS, 4)})
    total = sum(v["ms"] for v in out.values())
    cpu = None if args.no_cpu_baseline else cpu_baseline_small_ops(g, h, f, args.cpu_sample_edges)
    if cpu:
        cpu["gpu_ms_same_chain"] = round(sum(out[k]["ms"] for k in ("u_add_v", "u_add_v_backward", "edge_softmax", "edge_softmax_backward", "mhspmm",
                                                                    "mhspmm_transposed", "mhsddmm")), 3)
    return {"metric": "small per-edge operators on the C2 graph, ms per call, 1 MI355X", "value": round(total, 3), "unit": "ms (sum over the operators)",
            "n_gpus": 1, "steps": min(args.steps, 10), "warmup": 2, "ms_per_step": round(total, 3), "higher_is_better": False, "scaling": "weak",
            "vs_baseline": None, "dtype": "f32", "data": "synthetic",
            "config": {"workload": "small_ops_c2", "nodes": n, "edges": e, "heads": h, "out_feats": f}, "operators": out, "cpu_baseline": cpu}


def brief(rec):
    """The part of a workload's record that goes under "other_configs" of the default line."""
    keep = ("metric", "value", "unit", "ms_per_step", "config", "roofline", "roofline_bwd", "variants", "stash_variant", "fusescatter_pipeline", "sparse_fwd_bwd",
            "operators", "fused_sum_over_kernels", "hip_graph_replay", "knn_graph_ms", "backward_plain_scatter_us", "cpu_baseline", "peak_hbm_GiB")
    return {k: rec[k] for k in keep if k in rec}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--workload", default="gat_c2", choices=["gat_c2", "gat_c5", "gat_c5_l2", "gat_c5_train", "edgeconv_c3", "gmm_c4", "small_ops_c2", "gather_ceiling"])
    ap.add_argument("--no-others", action="store_true", help="gat_c2 only: do not append the other benchmark configurations to the line")
    ap.add_argument("--cpu-sample-edges", type=int, default=1_500_000)
    ap.add_argument("--no-cpu-baseline", action="store_true", help="skip the host-side baseline (profiling runs)")
    ap.add_argument("--permute-labels", action="store_true",
                    help="relabel the nodes of the R-MAT graphs by a random permutation (as Graph500 does): the generator puts the hubs at ids "
                         "that are sums of few powers of two, which costs the gathers of a graph larger than the caches 7-18 %% and helps the "
                         "small per-edge operators by up to 9 %%")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="also run a 1 GiB elementwise pass (torch.neg: reads 1 GiB, writes 1 GiB) so that profiler byte counters can be scaled")
    args = ap.parse_args()
    global PERMUTE_LABELS
    PERMUTE_LABELS = bool(args.permute_labels)
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures ONE GPU: the fused sparse-operator path is single-GPU (as is the reference); "
              "run with --gpus 1 (got --gpus %d, WORLD_SIZE=%s)" % (args.gpus, os.environ.get("WORLD_SIZE", "1")), file=sys.stderr)
        sys.exit(2)
    import torch
    if not torch.cuda.is_available():
        print("bench.py needs a GPU (torch.cuda.is_available() is False)", file=sys.stderr)
        sys.exit(2)
    if args.calibrate_copy:
        a = torch.empty(1 << 28, dtype=torch.float32, device="cuda:0").normal_()
        b = torch.empty_like(a)
        for _ in range(3):
            torch.neg(a, out=b)          # a kernel of its own name in the counter table (a plain copy_ shares hipMemcpy's)
        torch.cuda.synchronize()
        del a, b
    if args.workload == "gat_c2":
        rec = run_gat(args, 232965, 114_600_000, 256, 8, 32, "gat_c2")
        if not args.no_others:
            # the other benchmark configurations, each on its own graph, after this one's memory has been returned
            from ae_mlsys_gnn_amd import _lib
            import gc
            others = {}
            sub = argparse.Namespace(**vars(args))
            sub.steps, sub.warmup, sub.no_cpu_baseline = min(args.steps, 10), min(args.warmup, 3), True
            sub_cpu = argparse.Namespace(**vars(sub))          # a shorter host sample than the headline's: a few seconds
            sub_cpu.no_cpu_baseline, sub_cpu.cpu_sample_edges = args.no_cpu_baseline, min(args.cpu_sample_edges, 300_000)
            def train_with_permuted_labels():
                # the same step on the same graph with its node labels permuted at random (graphs.rmat_graph): times only, the
                # committed byte counts belong to the generator's labelling
                global PERMUTE_LABELS
                keep, PERMUTE_LABELS = PERMUTE_LABELS, True
                try:
                    r = run_gat_train(sub)
                finally:
                    PERMUTE_LABELS = keep
                return {"metric": r["metric"], "value": r["value"], "unit": r["unit"], "ms_per_step": r["ms_per_step"], "variants": r["variants"],
                        "config": dict(r["config"], node_labels="permuted at random (as Graph500 does to its generator's output)")}

            for name, fn in (("edgeconv_c3", lambda: run_edgeconv(args)), ("gmm_c4", lambda: run_gmm(args)),
                             ("gat_c5_layer1", lambda: run_gat(sub_cpu, 2449029, 61_900_000, 100, 8, 32, "gat_c5_layer1")),
                             ("gat_c5_train", lambda: run_gat_train(sub)), ("gat_c5_train_permuted_labels", train_with_permuted_labels),
                             ("small_ops_c2", lambda: run_small_ops(sub_cpu))):
                gc.collect()
                _lib.clear_schedule_cache()
                torch.cuda.empty_cache()
                torch.cuda.reset_peak_memory_stats()
                t0 = time.time()
                try:
                    others[name] = brief(fn())
                except Exception as exc:          # a failing side measurement must not take the headline with it
                    others[name] = {"error": "%s: %s" % (type(exc).__name__, exc)}
                others[name]["wall_s"] = round(time.time() - t0, 1)
            rec["other_configs"] = others
    elif args.workload == "gather_ceiling":
        rec = run_gather_ceiling(args)
    elif args.workload == "small_ops_c2":
        rec = run_small_ops(args)
    elif args.workload == "gat_c5":
        rec = run_gat(args, 2449029, 61_900_000, 100, 8, 32, "gat_c5_layer1")
    elif args.workload == "gat_c5_l2":          # the output layer of the C5 model alone: 256 -> 1 head x 47 classes (zero-padded to 48)
        rec = run_gat(args, 2449029, 61_900_000, 256, 1, 47, "gat_c5_layer2")
    elif args.workload == "gat_c5_train":
        rec = run_gat_train(args)
    elif args.workload == "edgeconv_c3":
        rec = run_edgeconv(args)
    else:
        rec = run_gmm(args)
    print(json.dumps(rec))


if __name__ == "__main__":
    main()
