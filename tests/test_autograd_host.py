"""The layers' backward passes on the CPU, the library calls replaced by the same computation in torch: what is tested is which operations
they record (gradients of gradients, on which gradient penalties train) and which passes over the edges they run."""
import pytest
import torch

from ae_mlsys_gnn_amd import graphs
from ae_mlsys_gnn_amd.operators.fused_gat import gat_dense_native
from ae_mlsys_gnn_amd.operators.fused_gmmconv import gmm_native


def _grads(loss, wrt, **kw):
    return torch.autograd.grad(loss, wrt, allow_unused=True, **kw)


@pytest.fixture
def gat_on_cpu(monkeypatch):
    def fold(W, al, ar, pad, want_all):
        fin, (_, h, f) = W.shape[0], al.shape
        wv = W.detach().view(fin, h, f)
        score = torch.cat([(wv * al).sum(-1), (wv * ar).sum(-1)], 1).detach()
        proj = torch.nn.functional.pad(wv, (0, pad)).reshape(fin, -1)
        return score.t().contiguous(), proj, torch.cat([proj, score], 1) if want_all else None

    def scores(feat, wt):
        s = feat.detach() @ wt.t()
        return s[:, :s.shape[1] // 2].contiguous(), s[:, s.shape[1] // 2:].contiguous()

    monkeypatch.setattr(gat_dense_native, "fold", staticmethod(fold))
    monkeypatch.setattr(gat_dense_native, "scores", staticmethod(scores))


@pytest.mark.parametrize("layout", ["contiguous", "transposed", "columns"])
def test_gat_projection_gradient_penalty(gat_on_cpu, layout):
    """d |dL/dW|^2 and d |dL/dattn|^2 by the input: exact for strided inputs as for contiguous ones."""
    from ae_mlsys_gnn_amd.layers.gatconv_layer import GATConv
    torch.manual_seed(1)
    m = GATConv(7, 5, 3).double()
    base = torch.randn(11, 7, dtype=torch.double)
    x = {"contiguous": base, "transposed": base.t().contiguous().t(), "columns": torch.cat([base, base], 1)[:, :7]}[layout].requires_grad_(True)
    c = [torch.randn(11, 3, 8, dtype=torch.double), torch.randn(11, 3, dtype=torch.double), torch.randn(11, 3, dtype=torch.double)]
    c[0][..., 5:] = 0
    params = [m.W, m.attn_l, m.attn_r]

    def composed(x):
        h = (x @ m.W).view(-1, 3, 5)
        return torch.nn.functional.pad(h, (0, 3)), (h * m.attn_l).sum(-1), (h * m.attn_r).sum(-1)

    result = []
    for f in (m._project, composed):
        loss = sum((o * w).sum() for o, w in zip(f(x), c))          # fixed gradients of the outputs: dL/dW is linear in x
        penalty = sum((g * g).sum() for g in _grads(loss, params, create_graph=True))
        result.append(_grads(penalty, [x])[0])
    assert torch.allclose(result[0], result[1], rtol=1e-12, atol=1e-12)


def _aggregate(row_ptr, col_ind, x, pseudo, mu, sigma):
    """sum over the edges of a row of w[p, k] * x[col_ind[p]] for x [N, F] or [N, K, F]: [N, K, F]."""
    w = torch.exp(-0.5 * (((pseudo.unsqueeze(1) - mu) * sigma) ** 2).sum(-1))
    rows = torch.repeat_interleave(torch.arange(row_ptr.numel() - 1), (row_ptr[1:] - row_ptr[:-1]).long())
    xs = x[col_ind.long()]
    msg = w.unsqueeze(-1) * (xs if xs.dim() == 3 else xs.unsqueeze(1))
    return torch.zeros(row_ptr.numel() - 1, *msg.shape[1:], dtype=x.dtype).index_add(0, rows, msg)


@pytest.fixture
def gmm_on_cpu(monkeypatch):
    """The library's GMMConv entry points in float64; `called` records which ones ran."""
    called = []

    def vjp(colptr, rowind, permute, x, pseudo, mu, sigma, grad_out):
        # in CSC order an edge's column is its source: gathers go the other way round, and the coordinates follow permute
        cols = torch.repeat_interleave(torch.arange(colptr.numel() - 1), (colptr[1:] - colptr[:-1]).long())
        order = torch.arange(rowind.numel()) if permute is None else permute.long()
        args = [t.detach().clone().requires_grad_(True) for t in (x, pseudo, mu, sigma)]
        w = torch.exp(-0.5 * (((args[1][order].unsqueeze(1) - args[2]) * args[3]) ** 2).sum(-1))
        xs, g = args[0][cols], grad_out.detach()[rowind.long()]
        xs, g = (t if t.dim() == 3 else t.unsqueeze(1) for t in (xs, g))
        return torch.autograd.grad((w.unsqueeze(-1) * xs * g).sum(), args)

    def shared(rowptr, colind, feat, pseudo, mu, sigma, *, pos_map=None, own_order=False):
        called.append("shared")
        return _aggregate(rowptr, colind, feat.detach(), pseudo.detach(), mu.detach(), sigma.detach())

    def shared_backward(colptr, rowind, permute, feat, pseudo, mu, sigma, grad_out, own_order=False):
        called.append("shared_backward")
        with torch.enable_grad():
            return vjp(colptr, rowind, permute, feat, pseudo, mu, sigma, grad_out)

    def backward(colptr, rowind, permute, node_feat, pseudo, mu, sigma, grad_out, sum_kernels=False, own_order=False):
        called.append("backward")
        with torch.enable_grad():
            return vjp(colptr, rowind, permute, node_feat, pseudo, mu, sigma, grad_out)

    monkeypatch.setattr(gmm_native, "gmmconv_shared", staticmethod(shared))
    monkeypatch.setattr(gmm_native, "gmmconv_shared_backward", staticmethod(shared_backward))
    monkeypatch.setattr(gmm_native, "gmmconv_backward", staticmethod(backward))
    return called


def _gmm_case(fin, fout, k, two, input_grad):
    from ae_mlsys_gnn_amd.layers.gmmconv_layer import GMMConv
    torch.manual_seed(2)
    g = graphs.add_csc_torch(graphs.rmat_graph(40, 300, seed=3))
    m = GMMConv(fin, fout, 2, k, bias=False).double()
    x = torch.randn(g.n, fin, dtype=torch.double, requires_grad=input_grad)
    ps = torch.rand(g.n_edges, 2, dtype=torch.double, requires_grad=True)
    run = lambda: m(g.row_ptr, g.col_ind, g.col_ptr, g.row_ind, g.permute, x, ps, ps[g.permute.long()] if two else None)

    def composed():
        agg = _aggregate(g.row_ptr, g.col_ind, x, ps, m.mu, m.inv_sigma)
        return torch.einsum("nkf,kof->no", agg, m.fc.weight.view(k, fout, fin))

    return m, x, ps, run, composed


@pytest.mark.parametrize("fin,fout,k", [(24, 9, 3), (24, 12, 3), (24, 40, 3)])
@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("input_grad", [False, True])
def test_gmm_gradient_penalty_on_the_weight(gmm_on_cpu, fin, fout, k, two, input_grad):
    """A penalty on dL/d(fc.weight) reaches the weight, the Gaussians, the coordinates and the input, in layers whose backward gathers
    their own gradient (the first two) as in the others."""
    m, x, ps, run, composed = _gmm_case(fin, fout, k, two, input_grad)
    wrt = [m.fc.weight, m.mu, m.inv_sigma, ps] + ([x] if input_grad else [])
    result = []
    for f in (run, composed):
        loss = (f() ** 2).sum()                     # the gradient of the output depends on everything, too
        gw = _grads(loss, [m.fc.weight], create_graph=True)[0]
        result.append((gw,) + _grads((gw * gw).sum(), wrt))
    for got, want in zip(*result):
        assert torch.allclose(got, want, rtol=1e-9, atol=1e-9 * float(want.detach().abs().max()))


@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("frozen", [False, True])
def test_gmm_frozen_gaussians_need_no_pass_over_the_edges(gmm_on_cpu, two, frozen):
    """With constant coordinates and input, the backward walks the edges for mu and inv_sigma only."""
    m, x, ps, run, composed = _gmm_case(24, 9, 3, two, False)
    ps.requires_grad_(False)
    m.mu.requires_grad_(not frozen)
    m.inv_sigma.requires_grad_(not frozen)
    run().sum().backward()
    assert gmm_on_cpu == (["shared"] if frozen else ["shared", "backward"])
    got = m.fc.weight.grad.clone()
    m.fc.weight.grad = None
    composed().sum().backward()
    assert torch.allclose(got, m.fc.weight.grad, rtol=1e-9, atol=1e-9)
