"""CPU-side checks of the host logic: the C ABI library loads and exports every declared symbol,
operators refuse to run without a GPU (no silent CPU fallback), graph builders are well formed."""
import ctypes
import os
import re

import pytest
import torch

from ae_mlsys_gnn_amd import _lib, graphs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _header_symbols():
    txt = open(os.path.join(ROOT, "include", "fgnn.h")).read()
    txt = re.sub(r"/\*.*?\*/", "", txt, flags=re.S)
    return sorted(set(re.findall(r"\b(fgnn_[a-z0-9_]+)\s*\(", txt)))


def test_library_exports_every_declared_symbol():
    assert os.path.exists(_lib.LIB_PATH), "libfgnn_hip.so has not been built (python -m ae_mlsys_gnn_amd.build)"
    names = _header_symbols()
    assert len(names) >= 29
    handle = ctypes.CDLL(_lib.LIB_PATH)
    missing = [n for n in names if not hasattr(handle, n)]
    assert not missing, "declared in include/fgnn.h but not exported: %s" % missing
    assert names == _lib.exported_symbols(), "ctypes signature table out of step with include/fgnn.h"
    assert _lib.lib().fgnn_version() >= 100


def test_only_the_c_abi_is_exported():
    import subprocess
    out = subprocess.run(["nm", "-D", "--defined-only", _lib.LIB_PATH], capture_output=True, text=True).stdout
    funcs = [l.split()[-1] for l in out.splitlines() if " T " in l]
    assert funcs and all(f.startswith("fgnn_") for f in funcs), [f for f in funcs if not f.startswith("fgnn_")]


def test_operators_refuse_cpu_tensors():
    from ae_mlsys_gnn_amd.operators import fused_gat, fused_edgeconv, fused_gmmconv
    g = graphs.add_csc_torch(graphs.uniform_graph(16, 40))
    x = torch.randn(16, 2, 4); a = torch.randn(16, 2)
    with pytest.raises(_lib.FgnnError):
        fused_gat.fused_gat_op(a, a, g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, 0.2, x)
    with pytest.raises(_lib.FgnnError):
        fused_edgeconv.fused_edgeconv_op(2, torch.zeros(32, dtype=torch.int32), torch.randn(16, 4), torch.randn(16, 4))
    with pytest.raises(_lib.FgnnError):
        fused_gmmconv.GaussianCp(torch.rand(5, 2), torch.rand(3, 2), torch.rand(3, 2))


def test_missing_library_fails_loudly(monkeypatch):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", os.path.join(ROOT, "does_not_exist.so"))
    with pytest.raises(_lib.FgnnError, match="missing"):
        _lib.lib()


def test_argument_errors_without_gpu():
    # argument validation happens before any launch, so the error codes are observable on a CPU box
    l = _lib.lib()
    assert l.fgnn_gat_forward(4, 4, 1, 4, None, None, None, None, 0.2, None, None, None, None, None, None, None, None, None, None, 0, None) == -1
    assert b"NULL" in l.fgnn_last_error()
    assert l.fgnn_edgeconv_forward(4, 4, 0, 2, None, None, None, None, None, None) == -2
    assert l.fgnn_mhsddmm(4, 4, 65, 4, None, None, None, None, None, None) == -4
    assert l.fgnn_csr2csc(-1, 4, 4, None, None, None, None, None, None, 0, None) == -2
    assert l.fgnn_schedule_num_items(None) == 0


def test_graph_builders():
    g = graphs.rmat_graph(500, 6000, seed=1)
    rp, ci = g.row_ptr.long(), g.col_ind.long()
    assert rp[0] == 0 and rp[-1] == g.n_edges and bool((rp[1:] >= rp[:-1]).all())
    dst = torch.repeat_interleave(torch.arange(g.n), rp[1:] - rp[:-1])
    keys = dst * g.n + ci
    assert bool((keys[1:] > keys[:-1]).all()), "edges must be unique and sorted by (dst, src)"
    assert int((dst == ci).sum()) == g.n, "exactly one self loop per node"
    assert g.n_edges == 6000 + g.n
    g2 = graphs.rmat_graph(500, 6000, seed=1)
    assert torch.equal(g.col_ind, g2.col_ind)
    deg = rp[1:] - rp[:-1]
    assert int(deg.max()) > 4 * float(deg.float().mean()), "R-MAT should be heavy tailed"
    # the same graph with its node labels permuted: a valid sorted CSR, the same in- and out-degree multisets, one self loop
    # per node, reproducible by seed, and the hubs no longer at the generator's ids
    gp = graphs.rmat_graph(500, 6000, seed=1, permute_labels=True)
    rpp, cip = gp.row_ptr.long(), gp.col_ind.long()
    dstp = torch.repeat_interleave(torch.arange(gp.n), rpp[1:] - rpp[:-1])
    kp = dstp * gp.n + cip
    assert gp.n_edges == g.n_edges and bool((kp[1:] > kp[:-1]).all()) and int((dstp == cip).sum()) == gp.n
    assert torch.equal(torch.sort(rpp[1:] - rpp[:-1]).values, torch.sort(deg).values)
    assert torch.equal(torch.sort(torch.bincount(cip, minlength=gp.n)).values, torch.sort(torch.bincount(ci, minlength=g.n)).values)
    assert torch.equal(gp.col_ind, graphs.rmat_graph(500, 6000, seed=1, permute_labels=True).col_ind)
    assert not torch.equal(rpp, rp)
    pts = torch.rand(3, 50, 3)
    src = graphs.knn_graph(pts, 7).view(3, 50, 7)
    assert bool((src[:, :, 0] == torch.arange(150).view(3, 50)).all()), "nearest neighbour of a point is itself"
    assert bool(((src // 50) == torch.arange(3).view(3, 1, 1)).all()), "neighbours stay inside the cloud"


def test_reference_import_recipe_resolves_to_this_package(tmp_path, monkeypatch):
    """The aliasing recipe documented for the reference tree: `operators` resolves to this package's
    mirror, so a layer file written against the reference's module names imports unchanged."""
    import importlib
    import sys
    import ae_mlsys_gnn_amd.operators as ops
    for name in ("operators", "operators.fused_gat", "operators.fused_edgeconv", "operators.fused_gmmconv", "operators.mhspmm",
                 "operators.edge_softmax", "operators.u_add_v", "operators.spmm", "operators.csr2csc"):
        monkeypatch.delitem(sys.modules, name, raising=False)
    monkeypatch.setitem(sys.modules, "operators", ops)
    for m in ("fused_gat", "fused_edgeconv", "fused_gmmconv", "mhspmm", "edge_softmax", "u_add_v", "spmm", "csr2csc"):
        monkeypatch.setitem(sys.modules, "operators." + m, getattr(ops, m))
    # a stand-in layer file using the reference's import lines (layers/gatconv_layer.py:7, edgeconv_layer.py:4,
    # gmmconv_layer.py:9-12)
    (tmp_path / "ref_style_layer.py").write_text(
        "from operators.fused_gat import fused_gat_op, fused_gat_stash_op, fused_gat_fusescatter\n"
        "from operators.fused_edgeconv import fused_edgeconv_op\n"
        "from operators.fused_gmmconv import GmmConvFuse, GmmConvStash, GaussianCp\n"
        "from operators.mhspmm import csrmhspmm\n"
        "from operators.edge_softmax import csr_edge_softmax\n"
        "from operators.u_add_v import u_add_v_op\n"
        "from operators.spmm import csrspmm\n"
        "from operators.csr2csc import sparsetrans\n")
    monkeypatch.syspath_prepend(str(tmp_path))
    mod = importlib.import_module("ref_style_layer")
    assert mod.fused_gat_op is ops.fused_gat.fused_gat_op and mod.sparsetrans is ops.csr2csc.sparsetrans


def test_reference_signatures_are_kept():
    """The public callables take the reference's arguments, by the same names and in the same order
    (operators/*.py, layers/*.py); anything this build adds comes after them and is optional."""
    import inspect
    from ae_mlsys_gnn_amd import layers, operators as ops
    want = {
        ops.fused_gat.fused_gat_op: "attn_row attn_col row_ptr col_ind col_ptr row_ind negative_slope in_feat save_memory",
        ops.fused_gat.fused_gat_stash_op: "attn_row attn_col row_ptr col_ind col_ptr row_ind negative_slope in_feat permute",
        ops.fused_gat.fused_gat_fusescatter: "attn_row attn_col row_ptr col_ind col_ptr row_ind negative_slope in_feat permute",
        ops.fused_edgeconv.fused_edgeconv_op: "k src_ind h_src h_dst",
        ops.fused_gmmconv.GmmConvFuse: "rowptr colind colptr rowind permute node_feat pseudo mu sigma",
        ops.fused_gmmconv.GmmConvStash: "rowptr colind colptr rowind permute node_feat pseudo mu sigma",
        ops.fused_gmmconv.GmmConvFuseEb: "rowptr colind colptr rowind permute node_feat pseudo mu sigma",
        ops.fused_gmmconv.GaussianCp: "pseudo mu sigma",
        ops.mhspmm.csrmhspmm: "rowptr colind colptr rowind permute feat attention",
        ops.edge_softmax.csr_edge_softmax: "rowptr h",
        ops.u_add_v.u_add_v_op: "row_ptr col_ind row_val col_val",
        ops.spmm.csrspmm: "rowptr colind x csr_data sym actnn",
        ops.csr2csc.sparsetrans: "rowptr colind numlist",
        layers.GATConv.forward: "self row_ptr col_ind col_ptr row_ind feat save_memory",
        layers.GATConv_stash.forward: "self row_ptr col_ind col_ptr row_ind feat permute",
        layers.EdgeConv.forward: "self k src_ind feat",
        layers.GMMConv.forward: "self rowptr colind colptr rowind permute feat pseudo",
        layers.GATConv.__init__: "self in_feats out_feats num_heads negative_slope",
        layers.EdgeConv.__init__: "self in_feat out_feat batch_norm allow_zero_in_degree",
        layers.GMMConv.__init__: "self in_feats out_feats dim n_kernels aggregator_type residual bias allow_zero_in_degree",
    }
    for fn, names in want.items():
        params = inspect.signature(fn).parameters
        ref = names.split()
        assert list(params)[:len(ref)] == ref, fn
        assert all(params[extra].default is not inspect.Parameter.empty for extra in list(params)[len(ref):]), fn


def test_more_argument_errors_without_gpu():
    l = _lib.lib()
    assert l.fgnn_knn_graph(1, 10, 3, 11, None, None, None) == -2                 # k > P
    assert l.fgnn_gather_rows(5, 0, None, None, None, None) == -2                 # W < 1
    assert l.fgnn_edge_softmax(-1, 0, 1, None, None, None, None) == -2
    assert l.fgnn_gaussian(4, 1, 2, None, None, None, None, None) == -1
    assert l.fgnn_coo2csr(4, 4, 3, None, None, 1, None, None, None, None, None, 0, None) == -1
    out = ctypes.c_void_p()
    assert l.fgnn_schedule_create(None, 4, 0, None, ctypes.byref(out)) == -1
    assert l.fgnn_schedule_create_bucketed(None, None, 4, 0, 0, 1, None, ctypes.byref(out)) == -1
    l.fgnn_schedule_destroy(None)                                                  # no-op on NULL


def test_gmm_backward_rule_stays_within_the_operator():
    """Every layer that the rule sends to the backward with the layer's own gradient is one that the library takes."""
    from ae_mlsys_gnn_amd.operators.fused_gmmconv import gmm_native, project_in_backward
    l = _lib.lib()
    for k in range(1, 6):
        for fin in (4, 64, 96, 128, 252, 256):
            if not gmm_native.shared_supported(k, fin):
                continue
            for fout in list(range(1, 70)) + [85, 86, 100, 127, 128, 129, 200, 255, 256, 257, 258, 300, 340, 341, 344, 352, 384, 512, 513]:
                for input_grad in (False, True):
                    if project_in_backward(k, fin, fout, input_grad, 10, 1000):
                        # pointers are missing, sizes are not refused
                        assert l.fgnn_gmm_backward(8, 8, k, 2, (fout + 3) // 4 * 4, *[None] * 8, 1, *[None] * 6, 0, None) == -1, (k, fin, fout)


@pytest.mark.parametrize("k,fin,fout,input_grad,degree,want", [
    (4, 256, 256, True, 15, False), (4, 256, 256, True, 20, True), (4, 256, 256, False, 3, True), (3, 128, 128, True, 9, False),
    (3, 128, 128, True, 15, True), (4, 256, 128, True, 4, False), (4, 256, 128, True, 9, True), (3, 128, 64, True, 4, True),
    (2, 16, 16, False, 50, True), (2, 16, 16, False, 200, False), (2, 32, 32, False, 260, False), (3, 32, 32, False, 260, True)])
def test_gmm_backward_rule_follows_the_degree(k, fin, fout, input_grad, degree, want):
    """Both sides of the lines that the degree draws (layer steps measured on either side)."""
    from ae_mlsys_gnn_amd.operators.fused_gmmconv import project_in_backward
    assert project_in_backward(k, fin, fout, input_grad, 100000, 100000 * degree) is want


def test_xcd_mapping_rule_without_gpu():
    """The rule behind the XCD-aware work lists: only a gfx950 device that shows all 256 compute units (eight XCDs of 32)
    is known to spread workgroups round-robin over eight XCDs; a partition of the part or another part gets plain lists."""
    l = _lib.lib()
    assert l.fgnn_xcd_mapping_for(b"gfx950:sramecc+:xnack-", 256) == 8
    assert l.fgnn_xcd_mapping_for(b"gfx950", 256) == 8
    assert l.fgnn_xcd_mapping_for(b"gfx950:sramecc+:xnack-", 128) == 0      # DPX: two devices of four XCDs
    assert l.fgnn_xcd_mapping_for(b"gfx950:sramecc+:xnack-", 32) == 0       # CPX: one XCD per device
    assert l.fgnn_xcd_mapping_for(b"gfx942:sramecc+:xnack-", 304) == 0
    assert l.fgnn_xcd_mapping_for(b"gfx9500", 256) == 0
    assert l.fgnn_xcd_mapping_for(None, 256) == 0
    assert l.fgnn_schedule_num_buckets(None) == 0


def test_column_sum_and_wide_row_argument_errors_without_gpu():
    l = _lib.lib()
    out = ctypes.c_void_p()
    assert l.fgnn_colsum_plan_create(None, None, 4, 4, 3, 8, 0, 0, None, ctypes.byref(out)) == -1
    assert l.fgnn_colsum_plan_create(None, None, 4, 4, 0, 8, 0, 0, None, None) == -1
    assert l.fgnn_edge_colsum(None, 8, None, None, None, 0, None) == -1
    assert l.fgnn_colsum_workspace_bytes(None, 8) == 0 and l.fgnn_colsum_plan_device_bytes(None) == 0
    l.fgnn_colsum_plan_destroy(None)
    assert l.fgnn_edge_rowsum(-1, 0, 8, None, None, None, None) == -2
    assert l.fgnn_u_add_v_backward_planned(4, 3, 8, None, None, None, None, None, None, None, 0, None) == -1
    # more than 1024 floats per head is the one width the GAT entries refuse; rows of many heads are grouped
    assert l.fgnn_gat_forward(4, 3, 2, 1028, None, None, None, None, 0.2, None, None, None, None, None, None, None, None, None, None, 0, None) == -4
    assert b"1024" in l.fgnn_last_error()
    assert l.fgnn_gat_forward(4, 3, 65, 4, None, None, None, None, 0.2, None, None, None, None, None, None, None, None, None, None, 0, None) == -4
    assert l.fgnn_mhsddmm(4, 3, 2, 1028, None, None, None, None, None, None) == -4
    # the workspace of a wide-row backward counts the head-group slices (and the stash slice when bit 1 is set)
    narrow = l.fgnn_gat_backward_workspace_bytes(1000, 4, 256, None, None, 0)
    wide = l.fgnn_gat_backward_workspace_bytes(1000, 8, 256, None, None, 0)
    assert wide > narrow + 5 * 1000 * 1024 * 4


# an input wider and narrower than the weights, a row or a column of them short, a bias that only broadcasts, one on another device
@pytest.mark.parametrize("x,w,b", [((4096, 128), (64, 64), None), ((4096, 50), (64, 64), None), ((4096, 64), (64,), None), ((4096, 64), (64, 64), (1,)),
                                   ((4096, 64), (64, 64), (63,)), ((4096, 64), (64, 64), (1, 64)), ((64,), (64, 64), None), ((4096, 64), (64, 64), "meta")])
def test_products_over_many_rows_take_only_what_fits(monkeypatch, x, w, b):
    """The kernels read by the sizes they are given: whatever does not fit stays with torch, which broadcasts or refuses it as it always did."""
    from ae_mlsys_gnn_amd.layers import dense
    from ae_mlsys_gnn_amd.operators import tall
    def no_kernel():
        raise AssertionError("a kernel was launched")
    monkeypatch.setattr(tall, "_plain", lambda *ts: True)
    monkeypatch.setattr(tall, "_matrices", lambda *ts: True)
    monkeypatch.setattr(tall, "lib", no_kernel)
    x, w = torch.randn(x), torch.randn(w)
    b = None if b is None else torch.empty(w.shape[0], device="meta") if b == "meta" else torch.randn(b)
    assert not tall.product_wanted(x, w, transposed=True, bias=b)
    if x.dim() == 2 and w.dim() == 2:
        with pytest.raises(_lib.FgnnError):
            tall.tall_product(x, w, transposed=True, bias=b)
    try:
        want = torch.matmul(x, w.t()) if b is None else torch.matmul(x, w.t()).add_(b)
    except RuntimeError:
        with pytest.raises(RuntimeError):
            dense.tall_linear(x, w, b)
    else:
        assert torch.equal(dense.tall_linear(x, w, b), want)


def test_products_over_many_rows_check_every_operand(monkeypatch):
    from ae_mlsys_gnn_amd.operators import tall
    monkeypatch.setattr(tall, "_plain", lambda *ts: True)
    monkeypatch.setattr(tall, "_matrices", lambda *ts: True)
    x, g = torch.randn(4096, 64), torch.randn(4096, 32)
    col = lambda n, h: (torch.randn(n, h), torch.randn(n, h))
    assert tall.product_wanted(x, torch.randn(64, 72), h_out=4) and tall.product_wanted(x, torch.randn(72, 64), h_in=4) and tall.reduce_wanted(x, g, 4)
    assert not tall.product_wanted(x, torch.randn(60, 72), h_out=4) and not tall.product_wanted(x, torch.randn(64, 64), h_in=4)
    assert not tall.reduce_wanted(x, g[:4000]) and not tall.reduce_wanted(x, g[:, 0])
    for extra in (None, col(4096, 3), col(4000, 4), (torch.randn(4096, 4), torch.randn(4096, 3)), (torch.randn(4096, 4).double(),) * 2, (torch.randn(4, 4096).t(),) * 2):
        with pytest.raises(_lib.FgnnError):
            tall.tall_product(x, torch.randn(72, 64), extra_in=extra)
        if extra is not None and extra[0].shape != (4096, 3):
            with pytest.raises(_lib.FgnnError):
                tall.tall_reduce(x, g, extra)
    with pytest.raises(_lib.FgnnError):
        tall.tall_reduce(x, g[:4000])


class _RecordingLib:
    """The library's work-list calls without a GPU: each call's name and its pointer arguments are kept."""

    def __init__(self):
        self.calls, self.made = [], 0

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, [a.value for a in args if isinstance(a, ctypes.c_void_p)]))
            if name.startswith("fgnn_schedule_create"):
                self.made += 1
                args[-1]._obj.value = self.made
            return 8 if name.endswith("num_buckets") else 0
        return call


@pytest.fixture
def lists_without_gpu(monkeypatch):
    import contextlib
    rec = _RecordingLib()
    monkeypatch.setattr(_lib, "lib", lambda: rec)
    monkeypatch.setattr(_lib, "_lib", rec)
    monkeypatch.setattr(_lib, "require_cuda", lambda *ts: None)
    monkeypatch.setattr(_lib, "device_guard", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(_lib, "stream_ptr", lambda: None)
    monkeypatch.setattr(_lib, "xcd_buckets_enabled", lambda *a: True)               # a skewed graph
    _lib.clear_schedule_cache()
    yield rec
    _lib.clear_schedule_cache()


def test_plain_lists_of_skewed_graphs_are_validated(lists_without_gpu, monkeypatch):
    """FGNN_VALIDATE=1: the ids are checked before the first gather by a plain list too, each index array of a pointer array by itself."""
    monkeypatch.setenv("FGNN_VALIDATE", "1")
    row_ptr, one, two = torch.tensor([0, 2, 3], dtype=torch.int32), torch.tensor([0, 1, 1], dtype=torch.int32), torch.tensor([1, 1, 0], dtype=torch.int32)
    checked = lambda: [args[1] for name, args in lists_without_gpu.calls if name == "fgnn_validate_graph"]
    for idx in (one, two, one):
        s = _lib.schedule_for(row_ptr, idx_tensor=idx, n_cols=2, flat=True)
        assert s.idx_tensor is None
    assert checked() == [one.data_ptr(), two.data_ptr()]
    one[0] = 1                                                                          # edited in place: checked again
    _lib.schedule_for(row_ptr, idx_tensor=one, n_cols=2, flat=True)
    assert checked() == [one.data_ptr(), two.data_ptr(), one.data_ptr()]


def test_own_order_lists_outlive_the_plain_lists_beside_them(lists_without_gpu):
    """Sixteen graphs with an own-order list a direction fit the cache, whatever plain lists their layers take besides; the plain
    lists are bounded, and one over an own-order list goes with it."""
    arrays = [[torch.tensor(v, dtype=torch.int32) for v in ([0, 2, 3], [0, 1, 1])] for _ in range(33)]
    for ptr, idx in arrays[:32]:
        _lib.edge_positions(ptr, idx)
    for _ in range(2):
        for ptr, idx in arrays[:32]:
            own = _lib.schedule_for(ptr, idx_tensor=idx, own_order=True)
            flat = _lib.schedule_for(ptr, idx_tensor=idx, own_order=True, flat=True)
            assert flat.flat_of is own and _lib.schedule_for(ptr, idx_tensor=idx, own_order=True, flat=True) is flat
    assert sum(name == "fgnn_schedule_create_flat" for name, _ in lists_without_gpu.calls) == 32         # built once each
    ptr, idx = arrays[0]
    assert _lib.schedule_for(ptr, idx_tensor=idx, flat=True) is _lib.schedule_for(ptr, idx_tensor=idx, flat=True)        # the caller's order
    for p, i in arrays[:32]:
        _lib.schedule_for(p, idx_tensor=i, own_order=True)
        _lib.schedule_for(p, idx_tensor=i, flat=True)
    assert len(_lib._flat_cache) <= 32 and len(_lib._sched_cache) <= 32
    base = _lib.schedule_for(ptr, idx_tensor=idx, own_order=True)
    _lib.schedule_for(ptr, idx_tensor=idx, own_order=True, flat=True)
    for p, i in arrays[1:32]:
        _lib.schedule_for(p, idx_tensor=i, own_order=True)
    _lib.edge_positions(*arrays[32])                                                    # one too many: the oldest goes, its plain list with it
    assert all(f.flat_of is not base for f in _lib._flat_cache.values())
    with pytest.raises(_lib.FgnnError):
        _lib.schedule_for(ptr, idx_tensor=idx, own_order=True)


@pytest.mark.parametrize("units", [256, 304, 80, 64])
def test_products_over_many_rows_launch_no_workgroup_past_the_compute_units(units):
    """A workgroup fills a unit's LDS, and the rows are dealt out over all of them: one too many doubles the time.  One to seven column ranges, with and
    without extra columns, few rows and many."""
    count = _lib.lib().fgnn_tall_product_workgroups
    for n in (1, 17, 4096, 65536, 70001, 169343, 2449029):
        for k, m, hin, hout in [(64, 64, 0, 0), (180, 384, 0, 6), (275, 256, 0, 4), (520, 128, 0, 1), (602, 64, 2, 0), (100, 256, 0, 8), (256, 100, 8, 0), (1024, 72, 0, 0),
                                (400, 512, 0, 0), (1024, 112, 0, 0), (16, 16, 0, 0)]:
            got = count(n, k, m, hin, hout, units)
            assert 0 < got <= units and got % 8 == 0, (n, k, m, got)
    assert count(70001, 2561, 16, 0, 0, units) == 0 and count(0, 16, 16, 0, 0, units) == 0


@pytest.mark.parametrize("n,degree,k,dim,row,aggregate,skewed,want", [
    (300000, 3, 4, 4, 100, False, False, False), (300000, 8, 3, 3, 128, False, False, False), (300000, 60, 4, 4, 128, False, False, True),
    (300000, 3, 2, 1, 256, False, False, False), (300000, 17, 2, 2, 256, False, False, True), (300000, 3, 2, 2, 256, False, True, True),
    (500000, 8, 3, 3, 96, True, False, False), (500000, 36, 3, 3, 96, True, True, True), (500000, 3, 4, 4, 64, False, False, False),
    (500000, 3, 4, 4, 16, False, False, True), (500000, 3, 3, 3, 64, True, False, True), (30000, 3, 4, 4, 128, False, False, True),
    (90000, 3, 3, 3, 128, False, True, True), (90000, 3, 3, 3, 128, False, False, False), (232965, 490, 2, 1, 16, False, True, True), (169343, 14, 3, 2, 64, False, True, True)])
def test_projected_coordinates_rule(n, degree, k, dim, row, aggregate, skewed, want):
    """The measured shapes: few edges a node, many sums and wide rows leave the projection to a pass of its own."""
    from ae_mlsys_gnn_amd.operators.fused_gmmconv import projected_pays
    assert projected_pays(n, n * degree, k, dim, row, aggregate, skewed) is want


def test_layer_asks_the_projection_rule(monkeypatch):
    """The rule gets the row that the layer's backward gathers: K x in floats where it aggregates first, else the output rounded up to 4."""
    from types import SimpleNamespace
    from ae_mlsys_gnn_amd.layers import GMMConv, GMMConv_stash, gmmconv_layer
    asked = []
    monkeypatch.setattr(gmmconv_layer, "projected_pays", lambda *a: asked.append(a) or False)
    monkeypatch.setattr(gmmconv_layer, "xcd_buckets_enabled", lambda *a: True)
    raw = SimpleNamespace(dtype=torch.float32, is_cuda=True, requires_grad=False)
    proj = SimpleNamespace(weight=raw, bias=raw)
    for layer, want in ((GMMConv(32, 40, 3, 3), (96, True)), (GMMConv(256, 41, 3, 3), (44, False)), (GMMConv_stash(32, 40, 3, 3), (40, False))):
        feat = torch.zeros(500, layer.fc.in_features, requires_grad=True)
        assert layer._projects(feat, raw, raw, proj, torch.zeros(501, dtype=torch.int32), torch.zeros(1000, dtype=torch.int32)) is False
        assert asked.pop() == (500, 1000, 3, 3, *want, True) and not asked


def test_products_over_many_rows_compile_whole():
    """Under torch.compile and torch.export the products are torch's, in one piece and for any number of rows."""
    from ae_mlsys_gnn_amd.layers import dense
    from ae_mlsys_gnn_amd.operators import tall
    x, w, b = torch.randn(5000, 64), torch.randn(48, 64), torch.randn(48)

    class Step(torch.nn.Module):
        def forward(self, t):
            return dense.tall_linear(t, w, b), dense.reduce_over_rows(t, t), dense.column_sum(t)

    class Linear(torch.nn.Module):
        def forward(self, t):
            return dense.tall_linear(t, w, b)
    with torch.no_grad():
        want = Step()(x)
        torch._dynamo.reset()
        got = torch.compile(Step(), backend="eager", fullgraph=True)(x)
        assert all(torch.equal(g, t) for g, t in zip(got, want))
        rows = torch.export.Dim("rows", min=2, max=1 << 22)
        for strict in (False, True):
            exported = torch.export.export(Linear(), (x,), dynamic_shapes=({0: rows},), strict=strict).module()
            assert exported(torch.randn(70000, 64)).shape == (70000, 48)
    torch._dynamo.reset()
    leaves = [t.clone().requires_grad_() for t in (x, w, b)]
    torch.compile(dense.tall_linear, backend="eager", fullgraph=True)(*leaves).sum().backward()
    assert all(t.grad is not None for t in leaves)
    torch._dynamo.reset()
    assert not tall._traced()
    seen = []
    torch.jit.trace(lambda t: (seen.append(tall._traced()), dense.tall_linear(t, w, b))[1], x, check_trace=False)
    assert seen == [True]


@pytest.mark.parametrize("ptr", [torch.tensor([0, 2, 3], dtype=torch.int32), torch.tensor([0, 2, 3])])
def test_row_lengths_are_read_from_the_gpu_only(monkeypatch, ptr):
    """The kernel that looks a pointer array over gets no host address and no other type; a layer with such an array says so."""
    from types import SimpleNamespace
    from ae_mlsys_gnn_amd.layers import GMMConv
    def no_kernel():
        raise AssertionError("a kernel was launched")
    monkeypatch.delenv("FGNN_XCD_BUCKETS", raising=False)
    monkeypatch.setattr(_lib, "lib", no_kernel)
    if ptr.dtype != torch.int32:
        monkeypatch.setattr(_lib, "require_cuda", lambda *ts: None)
    _lib.clear_schedule_cache()
    with pytest.raises(_lib.FgnnError):
        _lib.xcd_buckets_enabled(ptr, 3)
    raw = SimpleNamespace(dtype=torch.float32, is_cuda=True, requires_grad=False)
    with pytest.raises(_lib.FgnnError):
        GMMConv(64, 16, 1, 2)._projects(torch.zeros(2, 64), raw, raw, SimpleNamespace(weight=raw, bias=raw), ptr, torch.zeros(3, dtype=torch.int32))


def test_monet_projects_for_layers_that_do_not():
    """A layer of the caller's own, one that overrides the package's, a hooked one, and hooks on every module: the coordinates come projected, through
    the module."""
    from types import SimpleNamespace
    from ae_mlsys_gnn_amd.layers import GMMConv, GMMConv_stash
    from ae_mlsys_gnn_amd.train.train_gmmconv import MoNet, PseudoProj
    ps = SimpleNamespace(is_cuda=True, requires_grad=False)
    proj, seen = PseudoProj(2, 1), []

    class Own(torch.nn.Module):
        def __init__(self, *sizes):
            super().__init__()

        def forward(self, rowptr, colind, colptr, rowind, permute, feat, pseudo, pseudo_csc=None, own_order=False):
            seen.append((pseudo, pseudo_csc))
            return feat

    class Overridden(GMMConv):
        def forward(self, *args, **kwargs):
            return super().forward(*args, **kwargs)
    for c in (GMMConv, GMMConv_stash):
        assert proj.plain(c(8, 4, 1, 2), ps, ps)
    assert not proj.plain(Own(), ps, ps) and not proj.plain(Overridden(8, 4, 1, 2), ps, ps)
    hooked, patched = GMMConv(8, 4, 1, 2), GMMConv(8, 4, 1, 2)
    hooked.register_forward_pre_hook(lambda m, args: None)
    patched.forward = lambda *args, **kwargs: None
    assert not proj.plain(hooked, ps, ps) and not proj.plain(patched, ps, ps)
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, args, out: None)
    try:
        assert not proj.plain(GMMConv(8, 4, 1, 2), ps, ps)
    finally:
        handle.remove()
    model = MoNet(Own, 8, 4, 3, 0, 1, 2, 0.0)
    real = PseudoProj.forward
    try:
        PseudoProj.forward = lambda self, t: torch.ones(t.shape[0], 1)
        g = SimpleNamespace(row_ptr=None, col_ind=None, col_ptr=None, row_ind=None, permute=None)
        as_device = SimpleNamespace(is_cuda=True, requires_grad=False, shape=(6, 2))        # coordinates on the GPU, as far as the model can tell
        model(g, torch.rand(3, 8), as_device, pseudo_csc=as_device)
    finally:
        PseudoProj.forward = real
    assert len(seen) == 2 and all(torch.equal(t, torch.ones(6, 1)) for pair in seen for t in pair)


@pytest.mark.parametrize("n,k,m,product,reduction", [
    (16384, 64, 128, True, True), (49152, 256, 48, False, False), (57344, 64, 64, True, True), (65536, 64, 128, False, True), (65536, 128, 128, False, False),
    (65568, 128, 128, False, False), (65537, 128, 128, False, True), (122880, 256, 64, False, False), (131072, 64, 64, True, False), (131072, 128, 64, False, False),
    (131073, 128, 64, True, False), (169343, 384, 64, True, False), (169343, 256, 128, False, False), (169343, 64, 256, False, False), (262144, 128, 128, False, False),
    (524287, 128, 128, False, False), (524288, 64, 128, True, False), (700000, 64, 256, True, False), (700000, 602, 48, False, False)])
def test_products_over_many_rows_rules(monkeypatch, n, k, m, product, reduction):
    """The measured shapes, each at the form that a stream of calls runs faster with."""
    from ae_mlsys_gnn_amd.operators import tall
    monkeypatch.setattr(tall, "_plain", lambda *ts: True)
    x, g, w = (torch.empty(s, device="meta") for s in ((n, k), (n, m), (m, k)))
    assert tall.product_wanted(x, w, transposed=True) is product
    if m % 4 == k % 4 == 0:
        assert tall.reduce_wanted(x, g) is reduction


@pytest.mark.parametrize("entries,want", [(1, 1024), (1 << 22, 1024), (12 << 20, 1536), (115000000, 2048)])
def test_plain_lists_cut_hubs_by_the_size_of_the_graph(entries, want):
    assert _lib.flat_seg_len(entries) == want


@pytest.mark.parametrize("k,f,want", [(1, 4, True), (4, 16, True), (2, 28, True), (1, 64, True), (5, 12, False), (3, 20, False), (4, 12, True), (2, 36, False), (16, 4, True), (17, 4, False)])
def test_column_pass_batches(k, f, want):
    """Four rows or more in a batch: K times F, rounded up to a power of two, within the 64 floats of 16 lanes."""
    from ae_mlsys_gnn_amd.operators.fused_gmmconv import _column_pass_in_batches
    assert _column_pass_in_batches(k, f) is want
