"""The work lists (schedules) built on the device against the host-side builder they replace: item for item and
split for split the same list, for plain and XCD-aware lists, over segment lengths, bucket cut-offs and graph shapes
(empty rows, hubs, no edges at all, a single row); malformed pointer arrays are refused by both before any kernel
walks the index array with them."""
import math

import pytest
import torch

from tests.util import custom_graph, degree_edge_graph
from ae_mlsys_gnn_amd import graphs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _both(monkeypatch, ptr, idx, seg_len, min_deg, with_positions=True):
    from ae_mlsys_gnn_amd import _lib
    out = []
    for builder in ("device", "host"):
        monkeypatch.setenv("FGNN_SCHEDULE_BUILDER", builder)
        s = _lib.Schedule(ptr, seg_len, idx, min_deg, with_positions=with_positions)
        items, splits = s.export()
        pos = s.take_positions() if (idx is not None and with_positions) else None
        out.append((s.n_items, s.n_partials, s.n_edges, items.cpu(), splits.cpu(), None if pos is None else pos.cpu(), s.device_bytes(),
                    s.n_wave_slots, s.n_buckets))
    monkeypatch.delenv("FGNN_SCHEDULE_BUILDER")
    return out


GRAPHS = {
    "degrees": lambda: degree_edge_graph(n=700, seed=0),
    "rmat": lambda: graphs.rmat_graph(3000, 200000, seed=8),
    "uniform": lambda: graphs.uniform_graph(2000, 30000, seed=2),
    "no_edges": lambda: custom_graph([[], [], [], [], []]),
    "one_row": lambda: custom_graph([list(range(1)) * 700]),
    "hub_only": lambda: custom_graph([[0] * 5000, [], [1]]),
}


@pytest.mark.parametrize("name", sorted(GRAPHS))
@pytest.mark.parametrize("seg_len,min_deg", [(0, 0), (64, 16), (128, 16), (256, 64), (192, 100), (2048, 1)])
def test_device_built_schedules_equal_the_host_built_ones(name, seg_len, min_deg, monkeypatch):
    g = GRAPHS[name]().to(DEV)
    for idx in (None, g.col_ind):
        dev, host = _both(monkeypatch, g.row_ptr, idx, seg_len, min_deg)
        assert dev[:3] == host[:3], (name, "bucketed" if idx is not None else "plain", dev[:3], host[:3])
        assert torch.equal(dev[3], host[3]), "work items differ"
        assert torch.equal(dev[4], host[4]), "split tables differ"
        if idx is not None:
            assert torch.equal(dev[5], host[5]), "position maps differ"
        assert dev[6] == host[6]
        # the long items are a prefix of the list: nothing longer than 64 entries from slot n_wave_slots on, and the mark
        # is tight to the 64 slots (per source bucket) it is rounded up to
        for n_wave, n_buckets, items in ((dev[7], dev[8], dev[3]), (host[7], host[8], host[3])):
            length = (items[:, 2] - items[:, 1]) * (items[:, 0] >= 0)
            per = 64 * max(n_buckets, 1)
            assert 0 <= n_wave <= len(items) and (n_wave % per == 0 or n_wave == len(items))
            assert n_wave == len(items) or int(length[n_wave:].max()) <= 64
            if n_wave > 0:
                assert int(length[max(n_wave - per, 0):n_wave].max()) > 64 or n_wave == len(items)
            else:
                assert len(items) == 0 or int(length.max()) <= 64
        assert dev[7] == host[7]
        # the list covers every entry exactly once
        it = dev[3][dev[3][:, 0] >= 0].long()
        assert int((it[:, 2] - it[:, 1]).sum()) == g.n_edges


def test_malformed_pointer_arrays_are_refused_by_both_builders(monkeypatch):
    from ae_mlsys_gnn_amd import _lib
    g = graphs.rmat_graph(500, 20000, seed=3).to(DEV)
    dec = g.row_ptr.clone(); dec[100] = dec[101] + 5
    first = g.row_ptr.clone(); first[0] = 1
    for builder in ("device", "host"):
        monkeypatch.setenv("FGNN_SCHEDULE_BUILDER", builder)
        for bad, msg in ((dec, "decreases"), (first, r"ptr\[0\]")):
            for idx in (None, g.col_ind):
                with pytest.raises(_lib.FgnnError, match=msg):
                    _lib.Schedule(bad, 0, idx, 16)


@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_row_length_statistics(name):
    """The two numbers behind the choice of the work list (entries held by rows longer than the limit, the longest row)
    against torch reductions on the host."""
    import ctypes
    from ae_mlsys_gnn_amd import _lib
    g = GRAPHS[name]()
    deg = (g.row_ptr[1:] - g.row_ptr[:-1]).long()
    ptr_dev = g.row_ptr.to(DEV)
    for limit in (0, 1, 64, 512):
        stats = (ctypes.c_int64 * 2)()
        _lib.check(_lib.lib().fgnn_row_length_stats(_lib.ptr(ptr_dev), g.n, limit, ctypes.cast(stats, ctypes.c_void_p), _lib.stream_ptr()),
                   "fgnn_row_length_stats")
        assert int(stats[0]) == int(deg[deg > limit].sum()) and int(stats[1]) == int(deg.max() if g.n else 0)


def test_scheduled_sddmm_refuses_lists_it_cannot_use(monkeypatch):
    """fgnn_mhsddmm_scheduled stores its results at the caller's positions: a list of another graph and a list built
    without the position map are refused before any kernel runs; a list whose map was handed out stores in its own
    entry order."""
    from ae_mlsys_gnn_amd import _lib
    from ae_mlsys_gnn_amd._lib import lib, ptr, stream_ptr
    g = graphs.add_csc_torch(graphs.rmat_graph(500, 20000, seed=1)).to(DEV)
    other = graphs.rmat_graph(500, 20000, seed=2).to(DEV)
    n, h, f = g.n, 2, 8
    a = torch.randn(n, h, f, device=DEV)
    out = torch.empty(g.n_edges, h, device=DEV)

    def call(sched, graph=g):
        return lib().fgnn_mhsddmm_scheduled(n, graph.n_edges, h, f, ptr(graph.row_ptr), ptr(graph.col_ind), ptr(a), ptr(a), ptr(out), sched.handle,
                                            stream_ptr())
    good = _lib.Schedule(g.row_ptr, 0, g.col_ind, 16, with_positions=True)
    assert call(good) == 0
    plain = torch.empty_like(out)
    _lib.check(lib().fgnn_mhsddmm(n, g.n_edges, h, f, ptr(g.row_ptr), ptr(g.col_ind), ptr(a), ptr(a), ptr(plain), stream_ptr()), "fgnn_mhsddmm")
    assert torch.equal(out, plain)
    assert call(_lib.Schedule(other.row_ptr, 0, other.col_ind, 16, with_positions=True)) == -6
    assert b"another pointer array" in lib().fgnn_last_error()
    assert call(_lib.Schedule(g.row_ptr, 0, g.col_ind, 16, with_positions=False)) == -6
    assert b"edge positions" in lib().fgnn_last_error()
    taken = _lib.Schedule(g.row_ptr, 0, g.col_ind, 16, with_positions=True)
    pos = taken.take_positions()
    assert taken.n_buckets == 8 and not torch.equal(pos.cpu(), torch.arange(g.n_edges, dtype=torch.int32))
    assert call(taken) == 0
    assert torch.equal(out, plain[pos.long()])


def test_own_order_view_of_a_graph(monkeypatch):
    """_lib.own_order_view: the index array in the entry order of the CSR-side work list and the CSC-to-CSR map between the
    two entry orders.  Per-edge tensors kept in that order give the same multi-head SpMM (through the map) and SDDMM as the
    caller's order gives, bit for bit; rows keep their entries; the view is cached; plain lists give the arrays back."""
    from ae_mlsys_gnn_amd import _lib
    from ae_mlsys_gnn_amd.operators.mhspmm import mhsddmm, mhspmm
    monkeypatch.setenv("FGNN_XCD_BUCKETS", "1")
    monkeypatch.setenv("FGNN_BUCKET_MIN_DEG", "16")
    _lib.clear_schedule_cache()
    g = graphs.add_csc_torch(graphs.rmat_graph(1500, 90000, seed=5)).to(DEV)
    idx_own, perm_own = _lib.own_order_view(g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, g.permute)
    pos_r = _lib.edge_positions(g.row_ptr, g.col_ind)
    assert pos_r is not None and torch.equal(idx_own, g.col_ind[pos_r.long()])
    rows = torch.repeat_interleave(torch.arange(g.n, device=DEV), (g.row_ptr[1:] - g.row_ptr[:-1]).long())
    assert torch.equal(rows[pos_r.long()], rows)                       # a row's entries stay in the row
    assert torch.equal(torch.sort(perm_own).values, torch.arange(g.n_edges, dtype=torch.int32, device=DEV))
    again = _lib.own_order_view(g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, g.permute)
    assert again[0].data_ptr() == idx_own.data_ptr() and again[1].data_ptr() == perm_own.data_ptr()
    h, f = 4, 16
    torch.manual_seed(0)
    w = torch.randn(g.n_edges, h, device=DEV)
    a, b = torch.randn(g.n, h, f, device=DEV), torch.randn(g.n, h, f, device=DEV)
    w_own = w[pos_r.long()].contiguous()
    assert torch.equal(mhspmm(g.row_ptr, g.col_ind, w_own, a, own_order=True), mhspmm(g.row_ptr, g.col_ind, w, a))
    assert torch.equal(mhspmm(g.col_ptr, g.row_ind, w_own, a, pos_map=perm_own, own_order=True),
                       mhspmm(g.col_ptr, g.row_ind, w, a, pos_map=g.permute))
    assert torch.equal(mhsddmm(g.row_ptr, g.col_ind, a, b, own_order=True), mhsddmm(g.row_ptr, g.col_ind, a, b)[pos_r.long()])
    monkeypatch.setenv("FGNN_XCD_BUCKETS", "0")
    _lib.clear_schedule_cache()
    idx_p, perm_p = _lib.own_order_view(g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, g.permute)
    assert idx_p.data_ptr() == g.col_ind.data_ptr() and perm_p.data_ptr() == g.permute.data_ptr()
    _lib.clear_schedule_cache()


@pytest.mark.parametrize("private_names", [True, False])
def test_native_calls_follow_the_current_stream(monkeypatch, private_names):
    """The stream handed to the library is the current one of the tensors' device, with torch's private names and without them."""
    from ae_mlsys_gnn_amd import _lib
    if not private_names:
        monkeypatch.setattr(_lib, "_raw_stream", None)
        monkeypatch.setattr(_lib, "_DeviceGuard", None)
    dev = torch.device("cuda", torch.cuda.current_device())
    side = torch.cuda.Stream()
    with _lib.device_guard(dev):
        assert (_lib.stream_ptr().value or 0) == torch.cuda.current_stream().cuda_stream
        with torch.cuda.stream(side):
            assert _lib.stream_ptr().value == side.cuda_stream
    assert torch.cuda.current_device() == dev.index


def test_flat_list_over_bucketed_order(monkeypatch):
    """The plain list over an XCD-aware schedule's entry order: same operators, same per-edge order, its own cuts; positions stay put."""
    from ae_mlsys_gnn_amd import _lib
    from ae_mlsys_gnn_amd.operators import fused_gmmconv
    gmm_native = fused_gmmconv.gmm_native
    monkeypatch.setattr(fused_gmmconv, "_flat_list", lambda n, e, row, backward: row <= 64)         # the rule's sizes are too large for a test
    g = graphs.rmat_graph(3000, 400000, seed=3).to("cuda:0")
    base = _lib.Schedule(g.row_ptr, 0, g.col_ind, 0)
    if base.n_buckets == 0:
        pytest.skip("the device has no workgroup-to-XCD mapping: every list is plain")
    flat = _lib.Schedule(g.row_ptr, 128, flat_of=base)
    plain = _lib.Schedule(g.row_ptr, 128)
    assert flat.n_buckets == 0 and all(torch.equal(a, b) for a, b in zip(flat.export(), plain.export()))
    assert flat.device_bytes() == plain.device_bytes()
    with pytest.raises(_lib.FgnnError):
        base.take_positions()
    with pytest.raises(_lib.FgnnError):
        flat.take_positions()
    with pytest.raises(_lib.FgnnError):
        _lib.Schedule(g.row_ptr, 0, flat_of=flat)
    # own order: the narrow passes take the flat list, the wide ones the cut one, from the same per-edge copies
    pos = _lib.edge_positions(g.row_ptr, g.col_ind).long()
    ps = torch.rand(g.n_edges, 2, device="cuda:0")
    mu, sg = torch.zeros(2, 2, device="cuda:0"), torch.ones(2, 2, device="cuda:0")
    dst = torch.repeat_interleave(torch.arange(g.n, device="cuda:0"), (g.row_ptr[1:] - g.row_ptr[:-1]).long())
    w = torch.exp(-0.5 * (ps.double() ** 2).sum(1))
    assert _lib.schedule_for(g.row_ptr, idx_tensor=g.col_ind, own_order=True, flat=True).n_buckets == 0
    assert _lib.schedule_for(g.row_ptr, idx_tensor=g.col_ind, own_order=True).n_buckets > 0
    for f in (16, 64):
        x = torch.randn(g.n, 2, f, device="cuda:0")
        got = gmm_native.gmmconv(g.row_ptr, g.col_ind, x, ps[pos].contiguous(), mu, sg, sum_kernels=True, own_order=True)
        ref = torch.zeros(g.n, f, dtype=torch.float64, device="cuda:0").index_add_(0, dst, w[:, None] * x.sum(1).double()[g.col_ind.long()])
        mag = torch.zeros(g.n, f, dtype=torch.float64, device="cuda:0").index_add_(0, dst, w[:, None] * x.abs().sum(1).double()[g.col_ind.long()])
        assert bool(((got.double() - ref).abs() <= 64 * 2.0 ** -24 * mag + 1e-30).all())      # chains of at most 64, exp's last bits


# kernels past the summed pass' limit, rows past a wave, rows and base addresses off the 128-bit loads (those kernels add an item's entries to one chain),
# and two forms that do take the plain list
@pytest.mark.parametrize("k,f,off,summed", [(8, 32, 0, True), (5, 12, 0, True), (2, 16, 1, True), (2, 6, 0, True), (2, 16, 0, True), (2, 16, 2, False), (4, 16, 0, False), (3, 20, 0, False)])
def test_plain_list_costs_no_precision(monkeypatch, k, f, off, summed):
    """On a skewed graph large enough for the rule, the errors against float64 are no larger than with the list cut by source bucket."""
    from ae_mlsys_gnn_amd.operators import fused_gmmconv
    from ae_mlsys_gnn_amd.operators.csr2csc import csr2csc
    dev = "cuda:0"
    g = graphs.rmat_graph(20000, 4400000, seed=3, device=dev)
    g.col_ptr, g.row_ind, _ = csr2csc(g.row_ptr, g.col_ind)
    e = g.n_edges
    assert e >= 1 << 22
    gen = torch.Generator(device=dev).manual_seed(k * f)
    rnd = lambda *s: torch.rand(*s, generator=gen, device=dev)                # positive terms: nothing cancels, and what is lost is lost in the chains
    shifted = lambda *s: rnd(math.prod(s) + off)[off:].view(*s)
    x, go, ps = shifted(g.n, k, f), shifted(*((g.n, f) if summed else (g.n, k, f))), rnd(e, 1)
    mu, sg = torch.zeros(k, 1, device=dev), torch.full((k, 1), 0.5, device=dev)
    w = torch.exp(-0.5 * (0.5 * ps.double()) ** 2)                              # the weight of every kernel

    def gathered(ptr, idx, rows):
        out = torch.zeros(g.n, rows.shape[1], dtype=torch.float64, device=dev)
        dst = torch.repeat_interleave(torch.arange(g.n, device=dev), (ptr[1:] - ptr[:-1]).long())
        for i in range(0, e, 1 << 19):
            out.index_add_(0, dst[i:i + (1 << 19)], w[i:i + (1 << 19)] * rows[idx[i:i + (1 << 19)].long()].double())
        return out
    fwd = gathered(g.row_ptr, g.col_ind, x.sum(1) if summed else x.reshape(g.n, -1))
    bwd = gathered(g.col_ptr, g.row_ind, go.reshape(g.n, -1))

    def errors():
        out = fused_gmmconv.gmm_native.gmmconv(g.row_ptr, g.col_ind, x, ps, mu, sg, sum_kernels=summed)
        gx = fused_gmmconv.gmm_native.gmmconv_backward(g.col_ptr, g.row_ind, None, x, ps, mu, sg, go, sum_kernels=summed)[0]
        want = bwd[:, None, :].expand(g.n, k, f) if summed else bwd.view(g.n, k, f)
        return [float((a.double() - b).norm() / b.norm()) for a, b in ((out, fwd.view(out.shape)), (gx, want))]
    got = errors()
    monkeypatch.setattr(fused_gmmconv, "_flat_list", lambda *a: False)
    for a, b in zip(got, errors()):
        assert a <= 1.05 * b, (got, b)              # (the same kernel on the same list, or batches whose length does not grow with the item's)


def test_plain_list_of_a_skewed_graph_refuses_bad_ids(monkeypatch):
    """FGNN_VALIDATE=1 stops a bad id before the gather by the plain list as it does before the cut one's."""
    from ae_mlsys_gnn_amd import _lib
    from ae_mlsys_gnn_amd.operators import fused_gmmconv
    monkeypatch.setattr(fused_gmmconv, "_flat_list", lambda *a: True)
    monkeypatch.setenv("FGNN_VALIDATE", "1")
    g = graphs.rmat_graph(3000, 400000, seed=3).to("cuda:0")
    x, ps = torch.randn(g.n, 2, 16, device="cuda:0"), torch.rand(g.n_edges, 2, device="cuda:0")
    mu, sg = torch.zeros(2, 2, device="cuda:0"), torch.ones(2, 2, device="cuda:0")
    bad = g.col_ind.clone()
    bad[7] = g.n
    call = lambda idx: fused_gmmconv.gmm_native.gmmconv(g.row_ptr, idx, x, ps, mu, sg, sum_kernels=True)
    with pytest.raises(_lib.FgnnError, match="malformed graph"):
        call(bad)
    assert bool(torch.isfinite(call(g.col_ind)).all())
