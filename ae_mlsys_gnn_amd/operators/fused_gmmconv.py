"""Fused GMMConv (MoNet) operators: the reference's operators/fused_gmmconv.py surface on
libfgnn_hip.so.  The backward is one pass over the CSC arrays (the reference runs mhsddmm,
mhtranspose, a CSC gmmconv and GaussianBp: operators/fused_gmmconv.py:51-58) and implements the
closed-form Gaussian derivatives."""
from __future__ import annotations

import torch

from .._lib import FgnnError, as_f32, as_i32, check, device_guard, edge_positions, lib, ptr, require_cuda, schedule_for, stream_ptr, workspace
from .tall import product_wanted, tall_product


def _plain_list_for_summed_backward(n, e):
    """The summed backward gathers narrow rows ([N,F]); below an average degree of 64 it measured faster
    on the plain work list than on the XCD-aware one."""
    return e < 64 * n


def _flat_list(n, e, row, backward):
    """Whether a pass that gathers rows of `row` floats out of an [n, row] matrix takes the plain work list on skewed graphs too: rows
    narrower than a wave (which sums them batch by batch, so their length costs no precision) of a matrix that the eight L2s hold, or, in the
    backward, whose partial results are wider than what it gathers, twice that.  The cut by source bucket then has nothing to keep
    apart and only costs partial results (115 M edges, 233 k nodes, us, cut / plain: forward 16 x 2 floats, 30 MB 1590 / 1240, 48 floats, 45 MB
    2110 / 2280, 64 floats, 60 MB 2030 / 2430; backward of the sum, 16 floats 2630 / 1730, 64 floats, 60 MB 3750 / 2930; shared features, 32 floats
    2880 / 1770, 88 floats, 82 MB 4120 / 4770; 500 k nodes, 7 M edges, 2 x 16 floats 140 / 127 and 217 / 205).  Under 4 M edges either is as
    fast as often (169 k nodes, 2.3 M edges: 65 / 62, 68 / 78, 107 / 115)."""
    return e >= (1 << 22) and row <= 64 and row % 4 == 0 and 4 * n * row <= ((64 << 20) if backward else (32 << 20))


def _sums_in_batches(f, *arrays):
    """Whether a pass over rows no wider than a wave runs on the kernels that sum a row batch by batch, which take rows of F floats per mixture
    kernel as 128-bit loads.  The others add all entries of a list item to one chain (up to 2048 of them in a plain list; 8 kernels x 32 floats, error of
    the summed backward's input gradient, cut / plain: 20 k nodes, 4.4 M edges 2.5e-7 / 3.6e-7, 60 k, 30 M 4.2e-7 / 6.8e-7)."""
    return f % 4 == 0 and all(t is None or t.data_ptr() % 16 == 0 for t in arrays)


def _column_pass_in_batches(k, f):
    """Whether the column pass over rows of K x F floats has 16 lanes or fewer a row, each kernel's quarter of F rounded up to a power of two of them, and so
    four rows or more in a batch.  With two, the sums over the batches of an item of 2048 entries are a chain long enough to tell (5 kernels x 12
    floats, 17 M edges, error of the input gradient, cut / plain list: 6.0e-8 / 7.1e-8; 4 x 16 5.6e-8 / 5.3e-8)."""
    return f > 0 and k * max(4, 1 << (f - 1).bit_length()) <= 64


SUM_KERNELS_MAX = 4     # most mixture kernels that the summed column pass keeps in registers; with more, a pass over K x F floats


class gmm_native:
    """gmmconv.gmmconv / gmmconvstash / Gaussian / GaussianBp (src/fused_gmmconv/gmmconv.cc:36-94)."""

    @staticmethod
    def projection(proj, pseudo, k, dim, e):
        """(weight, bias) of a projection for pseudo [E, 2], checked; the operators form tanh(pseudo @ weight^T + bias) themselves."""
        weight, bias = as_f32(proj[0]), as_f32(proj[1])
        require_cuda(weight, bias)
        if tuple(weight.shape) != (dim, 2) or tuple(bias.shape) != (dim,) or tuple(pseudo.shape) != (e, 2) or not gmm_native.projection_supported(k, dim):
            raise FgnnError("gmmconv: projection weight %s, bias %s do not fit pseudo %s for K=%d dim=%d (at most 4 of each) E=%d" % (
                tuple(weight.shape), tuple(bias.shape), tuple(pseudo.shape), k, dim, e))
        return weight, bias

    @staticmethod
    def projection_supported(k, dim):
        return 0 < k <= 4 and 0 < dim <= 4

    @staticmethod
    def gmmconv(rowptr, colind, node_feat, pseudo, mu, sigma, *, pos_map=None, want_gauss=False, sum_kernels=False, own_order=False,
                bias=None, residual=None, proj=None):
        """bias [F] / residual [N,F] (with sum_kernels only): added to the summed output inside the operator's store.
        proj: (weight [dim,2], bias [dim]); pseudo is then [E,2] and the coordinates are tanh(pseudo @ weight^T + bias)."""
        require_cuda(rowptr, colind, node_feat, pseudo, mu, sigma, bias, residual)
        rowptr, colind = as_i32(rowptr), as_i32(colind)
        node_feat, pseudo, mu, sigma = as_f32(node_feat), as_f32(pseudo), as_f32(mu), as_f32(sigma)
        if node_feat.dim() != 3:
            raise FgnnError("node_feat must be [N,K,F], got %s" % (tuple(node_feat.shape),))
        n, k, f = node_feat.shape
        e = colind.numel()
        dim = mu.shape[1]
        pw, pb = (None, None) if proj is None else gmm_native.projection(proj, pseudo, k, dim, e)
        if mu.shape != (k, dim) or sigma.shape != (k, dim) or (proj is None and pseudo.shape != (e, dim)) or rowptr.numel() != n + 1:
            raise FgnnError("gmmconv: shape mismatch mu %s sigma %s pseudo %s for K=%d E=%d" % (
                tuple(mu.shape), tuple(sigma.shape), tuple(pseudo.shape), k, e))
        out = torch.empty((n, f), dtype=torch.float32, device=node_feat.device) if sum_kernels else torch.empty_like(node_feat)
        gauss = torch.empty((e, k), dtype=torch.float32, device=node_feat.device) if want_gauss else None
        epilogue = bias is not None or residual is not None
        if epilogue:
            if not sum_kernels:
                raise FgnnError("gmmconv: bias / residual are added to the sum over the kernels (sum_kernels=True)")
            bias = None if bias is None else as_f32(bias)
            residual = None if residual is None else as_f32(residual)
            if (bias is not None and tuple(bias.shape) != (f,)) or (residual is not None and tuple(residual.shape) != (n, f)):
                raise FgnnError("gmmconv: bias must be [%d] and residual [%d, %d]" % (f, n, f))
        # own_order: pseudo (and gauss) are indexed by the schedule's entry order, pseudo_caller[edge_positions(rowptr, colind)]
        flat = _flat_list(n, e, k * f, False) and _sums_in_batches(f, node_feat, bias, residual)
        sched = schedule_for(rowptr, idx_tensor=colind, own_order=own_order, n_cols=n, flat=flat)
        with device_guard(node_feat.device):
            ws, wsb = workspace(lib().fgnn_gmm_forward_workspace_bytes(sched.handle, k, f), node_feat.device)
            if proj is not None:
                check(lib().fgnn_gmm_forward_projected(n, e, k, dim, f, ptr(rowptr), ptr(colind), ptr(pos_map), ptr(node_feat), ptr(pseudo), ptr(pw), ptr(pb),
                                                       ptr(mu), ptr(sigma), ptr(bias), ptr(residual), ptr(out), ptr(gauss), int(sum_kernels), sched.handle,
                                                       ptr(ws), wsb, stream_ptr()), "fgnn_gmm_forward_projected")
            elif epilogue:
                check(lib().fgnn_gmm_forward_epilogue(n, e, k, dim, f, ptr(rowptr), ptr(colind), ptr(pos_map), ptr(node_feat), ptr(pseudo),
                                                      ptr(mu), ptr(sigma), ptr(bias), ptr(residual), ptr(out), ptr(gauss), sched.handle,
                                                      ptr(ws), wsb, stream_ptr()), "fgnn_gmm_forward_epilogue")
            else:
                check(lib().fgnn_gmm_forward(n, e, k, dim, f, ptr(rowptr), ptr(colind), ptr(pos_map), ptr(node_feat), ptr(pseudo),
                                             ptr(mu), ptr(sigma), ptr(out), ptr(gauss), int(sum_kernels), sched.handle, ptr(ws), wsb, stream_ptr()),
                      "fgnn_gmm_forward")
        return (out, gauss) if want_gauss else out

    @staticmethod
    def gmmconv_backward(colptr, rowind, permute, node_feat, pseudo, mu, sigma, grad_out, sum_kernels=False, own_order=False, proj=None):
        """(grad_feat, grad_pseudo, grad_mu, grad_sigma); with proj (see gmmconv) the gradients of its weight and bias in the place of
        grad_pseudo, and nothing is written per edge."""
        require_cuda(colptr, rowind, permute, node_feat, pseudo, mu, sigma, grad_out)
        colptr, rowind = as_i32(colptr), as_i32(rowind)
        permute = None if permute is None else as_i32(permute)      # None: pseudo / grad_pseudo in CSC order
        # raw pointers go to the kernels: contiguous copies of strided views, and every shape checked
        grad_out, node_feat, pseudo, mu, sigma = as_f32(grad_out), as_f32(node_feat), as_f32(pseudo), as_f32(mu), as_f32(sigma)
        if node_feat.dim() != 3 or mu.dim() != 2:
            raise FgnnError("gmmconv_backward: node_feat must be [N,K,F] and mu [K,dim], got %s and %s" % (tuple(node_feat.shape), tuple(mu.shape)))
        n, k, f = node_feat.shape
        e = rowind.numel()
        dim = mu.shape[1]
        dev = node_feat.device
        want_go = (n, f) if sum_kernels else (n, k, f)
        pw, pb = (None, None) if proj is None else gmm_native.projection(proj, pseudo, k, dim, e)
        if (mu.shape != (k, dim) or sigma.shape != (k, dim) or (proj is None and pseudo.shape != (e, dim)) or colptr.numel() != n + 1
                or tuple(grad_out.shape) != want_go or (permute is not None and permute.numel() != e)):
            raise FgnnError("gmmconv_backward: shape mismatch mu %s sigma %s pseudo %s grad_out %s col_ptr %d for N=%d K=%d F=%d E=%d" % (
                tuple(mu.shape), tuple(sigma.shape), tuple(pseudo.shape), tuple(grad_out.shape), colptr.numel(), n, k, f, e))
        grad_feat = torch.empty_like(node_feat)
        grad_pseudo = torch.empty((e, dim), dtype=torch.float32, device=dev) if proj is None else (torch.empty_like(pw), torch.empty_like(pb))
        grad_mu = torch.empty_like(mu)
        grad_sigma = torch.empty_like(sigma)
        # own_order: pseudo, grad_pseudo (and permute) are indexed by the schedule's entry order (gmm_edge_positions(colptr, rowind, True))
        summed = sum_kernels and k <= SUM_KERNELS_MAX
        flat = _flat_list(n, e, f if summed else k * f, True) and (summed or _column_pass_in_batches(k, f)) and _sums_in_batches(f, node_feat, grad_out)
        sched = schedule_for(colptr, idx_tensor=None if (sum_kernels and _plain_list_for_summed_backward(n, e)) else rowind, own_order=own_order, n_cols=n,
                             flat=flat)
        gmm_native._backward(n, e, k, dim, f, colptr, rowind, permute, node_feat, pseudo, (pw, pb), mu, sigma, grad_out, int(sum_kernels), grad_feat, grad_pseudo,
                             grad_mu, grad_sigma, sched, dev)
        return grad_feat, grad_pseudo, grad_mu, grad_sigma

    @staticmethod
    def _backward(n, e, k, dim, f, colptr, rowind, permute, feat, pseudo, proj, mu, sigma, grad_out, sum_kernels, grad_feat, grad_pseudo, grad_mu, grad_sigma, sched,
                  dev):
        with device_guard(dev):
            if proj[0] is None:
                ws, wsb = workspace(lib().fgnn_gmm_backward_workspace_bytes(sched.handle, k, dim, f), dev)
                check(lib().fgnn_gmm_backward(n, e, k, dim, f, ptr(colptr), ptr(rowind), ptr(permute), ptr(feat), ptr(pseudo),
                                              ptr(mu), ptr(sigma), ptr(grad_out), sum_kernels, ptr(grad_feat), ptr(grad_pseudo), ptr(grad_mu),
                                              ptr(grad_sigma), sched.handle, ptr(ws), wsb, stream_ptr()), "fgnn_gmm_backward")
                return
            ws, wsb = workspace(lib().fgnn_gmm_backward_projected_workspace_bytes(sched.handle, k, dim, f), dev)
            check(lib().fgnn_gmm_backward_projected(n, e, k, dim, f, ptr(colptr), ptr(rowind), ptr(permute), ptr(feat), ptr(pseudo), ptr(proj[0]), ptr(proj[1]),
                                                    ptr(mu), ptr(sigma), ptr(grad_out), sum_kernels, ptr(grad_feat), ptr(grad_pseudo[0]), ptr(grad_pseudo[1]),
                                                    ptr(grad_mu), ptr(grad_sigma), sched.handle, ptr(ws), wsb, stream_ptr()), "fgnn_gmm_backward_projected")

    @staticmethod
    def shared_supported(k, f):
        """Shapes the shared-feature (aggregate first) entry points take: the [N,f] rows as 128-bit slabs over
        at most a wave, the K accumulators in registers."""
        return f % 4 == 0 and 0 < f <= 256 and 0 < k <= 4

    @staticmethod
    def gmmconv_shared(rowptr, colind, feat, pseudo, mu, sigma, *, pos_map=None, own_order=False, proj=None):
        """out[i,k,:] = sum_p w[p,k] * feat[colind[p],:] for one [N,F] feature matrix shared by the K mixture
        kernels (the reference's gmmconv with node_feat[:,k,:] == feat for every k).  Returns [N,K,F]."""
        require_cuda(rowptr, colind, feat, pseudo, mu, sigma)
        rowptr, colind = as_i32(rowptr), as_i32(colind)
        feat, pseudo, mu, sigma = as_f32(feat), as_f32(pseudo), as_f32(mu), as_f32(sigma)
        if feat.dim() != 2:
            raise FgnnError("feat must be [N,F], got %s" % (tuple(feat.shape),))
        n, f = feat.shape
        k, dim = mu.shape
        e = colind.numel()
        pw, pb = (None, None) if proj is None else gmm_native.projection(proj, pseudo, k, dim, e)
        if sigma.shape != (k, dim) or (proj is None and pseudo.shape != (e, dim)) or rowptr.numel() != n + 1:
            raise FgnnError("gmmconv_shared: shape mismatch mu %s sigma %s pseudo %s for E=%d" % (
                tuple(mu.shape), tuple(sigma.shape), tuple(pseudo.shape), e))
        out = torch.empty((n, k, f), dtype=torch.float32, device=feat.device)
        sched = schedule_for(rowptr, idx_tensor=colind, own_order=own_order, n_cols=n, flat=_flat_list(n, e, f, False) and _sums_in_batches(f, feat))
        with device_guard(feat.device):
            ws, wsb = workspace(lib().fgnn_gmm_forward_workspace_bytes(sched.handle, k, f), feat.device)
            if proj is not None:
                check(lib().fgnn_gmm_forward_projected(n, e, k, dim, f, ptr(rowptr), ptr(colind), ptr(pos_map), ptr(feat), ptr(pseudo), ptr(pw), ptr(pb), ptr(mu),
                                                       ptr(sigma), None, None, ptr(out), None, 2, sched.handle, ptr(ws), wsb, stream_ptr()),
                      "fgnn_gmm_forward_projected (shared features)")
                return out
            check(lib().fgnn_gmm_forward(n, e, k, dim, f, ptr(rowptr), ptr(colind), ptr(pos_map), ptr(feat), ptr(pseudo),
                                         ptr(mu), ptr(sigma), ptr(out), None, 2, sched.handle, ptr(ws), wsb, stream_ptr()),
                  "fgnn_gmm_forward (shared features)")
        return out

    @staticmethod
    def gmmconv_shared_backward(colptr, rowind, permute, feat, pseudo, mu, sigma, grad_out, own_order=False, proj=None):
        """Backward of gmmconv_shared for grad_out [N,K,F]: (grad_feat [N,F], grad_pseudo (see gmmconv_backward), grad_mu, grad_sigma)."""
        require_cuda(colptr, rowind, permute, feat, pseudo, mu, sigma, grad_out)
        colptr, rowind = as_i32(colptr), as_i32(rowind)
        permute = None if permute is None else as_i32(permute)
        grad_out, feat, pseudo, mu, sigma = as_f32(grad_out), as_f32(feat), as_f32(pseudo), as_f32(mu), as_f32(sigma)
        if feat.dim() != 2 or mu.dim() != 2:
            raise FgnnError("gmmconv_shared_backward: feat must be [N,F] and mu [K,dim], got %s and %s" % (tuple(feat.shape), tuple(mu.shape)))
        n, f = feat.shape
        k, dim = mu.shape
        e = rowind.numel()
        dev = feat.device
        if grad_out.shape != (n, k, f):
            raise FgnnError("gmmconv_shared_backward: grad_out is %s, expected (%d, %d, %d)" % (tuple(grad_out.shape), n, k, f))
        pw, pb = (None, None) if proj is None else gmm_native.projection(proj, pseudo, k, dim, e)
        if sigma.shape != (k, dim) or (proj is None and pseudo.shape != (e, dim)) or colptr.numel() != n + 1 or (permute is not None and permute.numel() != e):
            raise FgnnError("gmmconv_shared_backward: shape mismatch sigma %s pseudo %s col_ptr %d for N=%d K=%d E=%d" % (
                tuple(sigma.shape), tuple(pseudo.shape), colptr.numel(), n, k, e))
        parts = torch.empty((n, k, f), dtype=torch.float32, device=dev)      # kernel k's share of grad_feat
        grad_pseudo = torch.empty((e, dim), dtype=torch.float32, device=dev) if proj is None else (torch.empty_like(pw), torch.empty_like(pb))
        grad_mu = torch.empty_like(mu)
        grad_sigma = torch.empty_like(sigma)
        # same work list as the summed backward, so that one CSC-side copy of own-order edge data serves both kinds of layer
        sched = schedule_for(colptr, idx_tensor=None if _plain_list_for_summed_backward(n, e) else rowind, own_order=own_order, n_cols=n,
                             flat=_flat_list(n, e, k * f, True) and _column_pass_in_batches(k, f) and _sums_in_batches(f, feat, grad_out))
        gmm_native._backward(n, e, k, dim, f, colptr, rowind, permute, feat, pseudo, (pw, pb), mu, sigma, grad_out, 2, parts, grad_pseudo, grad_mu, grad_sigma, sched,
                             dev)
        return parts.sum(1), grad_pseudo, grad_mu, grad_sigma

    @staticmethod
    def Gaussian(pseudo, mu, sigma):
        require_cuda(pseudo, mu, sigma)
        pseudo, mu, sigma = as_f32(pseudo), as_f32(mu), as_f32(sigma)
        e, dim = pseudo.shape
        k = mu.shape[0]
        out = torch.empty((e, k), dtype=torch.float32, device=pseudo.device)
        with device_guard(pseudo.device):
            check(lib().fgnn_gaussian(e, k, dim, ptr(pseudo), ptr(mu), ptr(sigma), ptr(out), stream_ptr()), "fgnn_gaussian")
        return out

    @staticmethod
    def GaussianBp(pseudo, mu, sigma, grad_out):
        require_cuda(pseudo, mu, sigma, grad_out)
        pseudo, mu, sigma, grad_out = as_f32(pseudo), as_f32(mu), as_f32(sigma), as_f32(grad_out)
        e, dim = pseudo.shape
        k = mu.shape[0]
        gp = torch.empty_like(pseudo)
        gm = torch.empty_like(mu)
        gs = torch.empty_like(sigma)
        with device_guard(pseudo.device):
            ws, wsb = workspace(lib().fgnn_gaussian_backward_workspace_bytes(e, k, dim), pseudo.device)
            check(lib().fgnn_gaussian_backward(e, k, dim, ptr(pseudo), ptr(mu), ptr(sigma), ptr(grad_out), ptr(gp), ptr(gm),
                                               ptr(gs), ptr(ws), wsb, stream_ptr()), "fgnn_gaussian_backward")
        return gp, gm, gs


def _epilogue_grads(ctx, grad_out, first):
    """Gradients of the optional (bias, residual) inputs at positions first, first + 1 of a Function's inputs."""
    from ..layers.dense import column_sum
    gb = column_sum(grad_out) if (ctx.has_bias and ctx.needs_input_grad[first]) else None
    gr = grad_out if (ctx.has_res and ctx.needs_input_grad[first + 1]) else None
    return gb, gr


def GmmConvFuse(rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma):
    return GmmFuseFunction.apply(rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma)


class GmmFuseFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma):
        out = gmm_native.gmmconv(rowptr, colind, node_feat, pseudo, mu, sigma)      # [N, K, F]
        ctx.save_for_backward(rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma = ctx.saved_tensors
        grad_feat, grad_pseudo, grad_mu, grad_sigma = gmm_native.gmmconv_backward(
            colptr, rowind, permute, node_feat, pseudo, mu, sigma, grad_out.contiguous())
        return None, None, None, None, None, grad_feat, grad_pseudo, grad_mu, grad_sigma


def GmmConvFuseSum(rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma, bias=None, residual=None):
    """GmmConvFuse(...).sum(1) as one operator: the sum over the K mixture kernels is fused into the
    forward's store and the backward gathers [N,F] gradient rows.  Returns [N,F].
    bias [F], residual [N,F] (optional): the rest of the layer's forward (layers/gmmconv_layer.py:69-75), added in
    the same store."""
    return GmmFuseSumFunction.apply(rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma, bias, residual)


def GmmConvFuseSumTwoOrders(rowptr, colind, colptr, rowind, node_feat, pseudo_csr, pseudo_csc, mu, sigma, own_order=False, bias=None,
                            residual=None):
    """GmmConvFuseSum for a caller that has the pseudo-coordinates in both edge orders
    (pseudo_csc == pseudo_csr[permute], e.g. the same elementwise projection applied to constant
    edge data stored both ways).  The forward reads pseudo_csr, the backward reads pseudo_csc and
    returns its gradient in CSC order: no per-edge gather or scatter through permute.  pseudo_csr
    gets no gradient; the caller's parameters receive theirs through pseudo_csc (None: forward only).
    own_order: the two tensors are in the entry order of the operators' own schedules,
    pseudo_csr[gmm_edge_positions(rowptr, colind)] and pseudo_csc[gmm_edge_positions(colptr, rowind, True)]:
    every pass then streams its per-edge data."""
    if pseudo_csc is None:
        return gmm_native.gmmconv(rowptr, colind, node_feat, pseudo_csr, mu, sigma, sum_kernels=True, own_order=own_order, bias=bias,
                                  residual=residual)
    return GmmFuseSumTwoOrdersFunction.apply(rowptr, colind, colptr, rowind, node_feat, pseudo_csr, pseudo_csc, mu, sigma, own_order, bias, residual)


def GmmConvStashSumTwoOrders(rowptr, colind, colptr, rowind, node_feat, pseudo_csr, pseudo_csc, mu, sigma, own_order=False, bias=None,
                             residual=None):
    """The stash variant with the pseudo-coordinates in both edge orders: as GmmConvFuseSumTwoOrders, and the
    forward also writes the Gaussian weights [E,K] (in the order of pseudo_csr) and keeps them until the
    backward, the memory cost of the reference's stash variant (operators/fused_gmmconv.py:100-118).  The
    backward is the same single pass: recomputing a weight is cheaper than reading it back through a
    transposition."""
    return GmmStashSumTwoOrdersFunction.apply(rowptr, colind, colptr, rowind, node_feat, pseudo_csr, pseudo_csc, mu, sigma, own_order, bias, residual)


class GmmStashSumTwoOrdersFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rowptr, colind, colptr, rowind, node_feat, pseudo_csr, pseudo_csc, mu, sigma, own_order, bias=None, residual=None):
        out, gauss = gmm_native.gmmconv(rowptr, colind, node_feat, pseudo_csr, mu, sigma, want_gauss=True, sum_kernels=True,
                                        own_order=own_order, bias=bias, residual=residual)
        ctx.save_for_backward(colptr, rowind, node_feat, pseudo_csc, mu, sigma, gauss)
        ctx.own_order = own_order
        ctx.has_bias, ctx.has_res = bias is not None, residual is not None
        return out

    @staticmethod
    def backward(ctx, grad_out):
        colptr, rowind, node_feat, pseudo_csc, mu, sigma, _gauss = ctx.saved_tensors
        grad_feat, grad_pseudo_csc, grad_mu, grad_sigma = gmm_native.gmmconv_backward(
            colptr, rowind, None, node_feat, pseudo_csc, mu, sigma, grad_out.contiguous(), sum_kernels=True, own_order=ctx.own_order)
        return (None, None, None, None, grad_feat, None, grad_pseudo_csc, grad_mu, grad_sigma, None) + _epilogue_grads(ctx, grad_out.contiguous(), 10)


def gmm_edge_positions(ptr_arr, idx, summed_backward=False):
    """int32 [E] (or None = identity): caller's position of every entry in the order in which the GMMConv
    operators walk (ptr_arr, idx) when called with own_order=True.  summed_backward: for the (col_ptr,
    row_ind) arrays of the layers' backward passes (GmmConvFuseSumTwoOrders, GmmAggregateTwoOrders), which
    keep the caller's order on graphs of low average degree."""
    require_cuda(ptr_arr, idx)
    ptr_arr, idx = as_i32(ptr_arr), as_i32(idx)
    if summed_backward and _plain_list_for_summed_backward(ptr_arr.numel() - 1, idx.numel()):
        schedule_for(ptr_arr)
        return None
    return edge_positions(ptr_arr, idx)


class GmmFuseSumTwoOrdersFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rowptr, colind, colptr, rowind, node_feat, pseudo_csr, pseudo_csc, mu, sigma, own_order, bias=None, residual=None):
        out = gmm_native.gmmconv(rowptr, colind, node_feat, pseudo_csr, mu, sigma, sum_kernels=True, own_order=own_order, bias=bias,
                                 residual=residual)      # [N, F]
        ctx.save_for_backward(colptr, rowind, node_feat, pseudo_csc, mu, sigma)
        ctx.own_order = own_order
        ctx.has_bias, ctx.has_res = bias is not None, residual is not None
        return out

    @staticmethod
    def backward(ctx, grad_out):
        colptr, rowind, node_feat, pseudo_csc, mu, sigma = ctx.saved_tensors
        grad_feat, grad_pseudo_csc, grad_mu, grad_sigma = gmm_native.gmmconv_backward(
            colptr, rowind, None, node_feat, pseudo_csc, mu, sigma, grad_out.contiguous(), sum_kernels=True, own_order=ctx.own_order)
        return (None, None, None, None, grad_feat, None, grad_pseudo_csc, grad_mu, grad_sigma, None) + _epilogue_grads(ctx, grad_out.contiguous(), 10)


def GmmAggregate(rowptr, colind, colptr, rowind, permute, feat, pseudo, mu, sigma):
    """Aggregate first: agg[i,k,:] = sum_p w[p,k] * feat[colind[p],:] for feat [N,F] -> [N,K,F].  A GMMConv
    layer whose input is narrower than K x its output multiplies by the fc weights afterwards
    (sum_k agg[:,k,:] @ W_k equals the reference's sum over k of the aggregated fc(feat)[:,k,:]), so an
    edge gathers F floats instead of K x out."""
    return GmmAggregateFunction.apply(rowptr, colind, colptr, rowind, permute, feat, pseudo, mu, sigma)


class GmmAggregateFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rowptr, colind, colptr, rowind, permute, feat, pseudo, mu, sigma):
        out = gmm_native.gmmconv_shared(rowptr, colind, feat, pseudo, mu, sigma)
        ctx.save_for_backward(colptr, rowind, permute, feat, pseudo, mu, sigma)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        colptr, rowind, permute, feat, pseudo, mu, sigma = ctx.saved_tensors
        grad_feat, grad_pseudo, grad_mu, grad_sigma = gmm_native.gmmconv_shared_backward(
            colptr, rowind, permute, feat, pseudo, mu, sigma, grad_out.contiguous())
        return None, None, None, None, None, grad_feat, grad_pseudo, grad_mu, grad_sigma


def GmmAggregateTwoOrders(rowptr, colind, colptr, rowind, feat, pseudo_csr, pseudo_csc, mu, sigma, own_order=False):
    """GmmAggregate for a caller that has the pseudo-coordinates in both edge orders (see
    GmmConvFuseSumTwoOrders; pseudo_csc None: forward only)."""
    if pseudo_csc is None:
        return gmm_native.gmmconv_shared(rowptr, colind, feat, pseudo_csr, mu, sigma, own_order=own_order)
    return GmmAggregateTwoOrdersFunction.apply(rowptr, colind, colptr, rowind, feat, pseudo_csr, pseudo_csc, mu, sigma, own_order)


class GmmAggregateTwoOrdersFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rowptr, colind, colptr, rowind, feat, pseudo_csr, pseudo_csc, mu, sigma, own_order):
        out = gmm_native.gmmconv_shared(rowptr, colind, feat, pseudo_csr, mu, sigma, own_order=own_order)
        ctx.save_for_backward(colptr, rowind, feat, pseudo_csc, mu, sigma)
        ctx.own_order = own_order
        return out

    @staticmethod
    def backward(ctx, grad_out):
        colptr, rowind, feat, pseudo_csc, mu, sigma = ctx.saved_tensors
        grad_feat, grad_pseudo_csc, grad_mu, grad_sigma = gmm_native.gmmconv_shared_backward(
            colptr, rowind, None, feat, pseudo_csc, mu, sigma, grad_out.contiguous(), own_order=ctx.own_order)
        return None, None, None, None, grad_feat, None, grad_pseudo_csc, grad_mu, grad_sigma, None


def GmmProjectedTwoOrders(rowptr, colind, colptr, rowind, node_feat, raw_csr, raw_csc, weight, bias, mu, sigma, own_order=False, keep_gauss=False,
                          out_bias=None, residual=None):
    """GmmConvFuseSumTwoOrders (node_feat [N,K,F]; keep_gauss: GmmConvStashSumTwoOrders) or GmmAggregateTwoOrders (node_feat [N,F]) on the
    coordinates tanh(raw @ weight^T + bias) of constant raw [E,2] edge data, in both edge orders: the passes over the edges form them
    themselves, and the backward sums the gradients of weight, bias, mu and sigma where it forms the derivatives of the mixture weights.
    Instead of 4 E dim floats of coordinates and their gradients and E K of derivatives, written and read back, an edge costs 8 bytes
    a pass (115 M edges, 2 kernels of 1 coordinate, two layers: MoNet step 8.96 -> 7.64 ms)."""
    return GmmProjectedTwoOrdersFunction.apply(rowptr, colind, colptr, rowind, node_feat, raw_csr, raw_csc, weight, bias, mu, sigma, own_order, keep_gauss,
                                               out_bias, residual)


class GmmProjectedTwoOrdersFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rowptr, colind, colptr, rowind, node_feat, raw_csr, raw_csc, weight, bias, mu, sigma, own_order, keep_gauss, out_bias=None, residual=None):
        gauss = None
        if node_feat.dim() == 2:
            out = gmm_native.gmmconv_shared(rowptr, colind, node_feat, raw_csr, mu, sigma, own_order=own_order, proj=(weight, bias))
        else:
            out = gmm_native.gmmconv(rowptr, colind, node_feat, raw_csr, mu, sigma, want_gauss=keep_gauss, sum_kernels=True, own_order=own_order, bias=out_bias,
                                     residual=residual, proj=(weight, bias))
            out, gauss = out if keep_gauss else (out, None)
        ctx.save_for_backward(colptr, rowind, node_feat, raw_csc, weight, bias, mu, sigma, gauss)
        ctx.own_order = own_order
        ctx.has_bias, ctx.has_res = out_bias is not None, residual is not None
        return out

    @staticmethod
    def backward(ctx, grad_out):
        colptr, rowind, node_feat, raw_csc, weight, bias, mu, sigma, _gauss = ctx.saved_tensors
        args = (colptr, rowind, None, node_feat, raw_csc, mu, sigma, grad_out.contiguous())
        if node_feat.dim() == 2:
            grads = gmm_native.gmmconv_shared_backward(*args, own_order=ctx.own_order, proj=(weight, bias))
        else:
            grads = gmm_native.gmmconv_backward(*args, sum_kernels=True, own_order=ctx.own_order, proj=(weight, bias))
        grad_feat, (grad_w, grad_b), grad_mu, grad_sigma = grads
        return (None, None, None, None, grad_feat, None, None, grad_w, grad_b, grad_mu, grad_sigma, None, None) + _epilogue_grads(ctx, grad_out.contiguous(), 13)


def projected_pays(n, e, k, dim, row, aggregate, skewed):
    """Whether the passes over the edges that project the coordinates themselves are no slower than projecting them beforehand, for n nodes, e edges and
    a backward that gathers rows of `row` floats (aggregate: of the layer that aggregates its input first).  What they save is per edge; the
    sums of the parameters' gradients, 2 K dim + 3 dim of them in LDS, cost every wave its start and end, and a wave on rows wider than 64
    floats has one node's edges.  (us of a layer's forward and backward, formed beforehand / in the passes, 300 k nodes, uniform: 128 floats,
    5 sums, degree 3 754 / 867, 17 1189 / 1160; 15 sums, degree 8 912 / 1106, 25 1620 / 1551; 44 sums, degree 8 2202 / 2967, 61 ahead; 256
    floats, 14 sums, degree 8 1.04 of it, 17 0.98; 64 floats, 44 sums, degree 5 1.08, 12 0.95; aggregated rows of 96 floats, 27 sums, degree 3
    1.4, 21 1.05, 36 0.96.  On skewed graphs half of the columns are nearly empty, and the copies cost more: 256 floats 0.90 to 1.0.)  Few nodes are
    bound by the host, which the copies' launches cost 45 us."""
    sums = 2 * k * dim + 3 * dim
    if row <= 32 or n < 65536 or n * sums < (1 << (22 if skewed else 20)):
        return True
    if row <= 64:                           # lane groups: 4 or more nodes a wave
        return aggregate or e >= n * (sums - 10) / 4
    least = (10 + sums) * (0.6 if aggregate else 1.0)
    if row > 128:
        if skewed and sums <= 30:
            return True
        least /= 2
    return e >= n * least


def project_in_backward(k, fin, fout, input_grad, n, e):
    """Which rows the backward of an aggregate-first layer (n nodes, e edges) gathers per edge: K x fin floats, the gradient of the aggregate,
    or the fout floats (rounded up to 4) of the layer's own gradient, for the price of projecting the input again (and of one more
    product for the input's gradient).  Layer steps, gathering K x fin / fout floats: 169 k nodes, 2.3 M edges, 384 / 64 floats 1.69 ->
    1.01 ms (1.16 with the input's gradient), 128 / 64 0.76 -> 0.68 (0.74), 96 / 44 0.66 -> 0.66 (0.69), 128 / 84 0.78 -> 0.89 ms (0.99);
    300 k nodes, 0.9 M edges, 256 / 100 floats 1.53 -> 1.49 (1.70): the lines lie at ratios of 2 and 3.
    With the input's gradient and few edges the products, n fin K fout multiply-adds more, outweigh the gathers, at about 20 of them for
    every float that an edge no longer gathers: 169 k nodes of 15 edges, 1024 / 256 floats 5.47 -> 5.56 ms, 1024 / 128 4.47 -> 3.16;
    300 k nodes of 4 edges, 1024 / 128 4.21 -> 4.20, 384 / 64 1.54 -> 1.46.  On dense graphs rows of up to two cache lines cost what
    rows of one do: 32 / 16 floats 0.95 -> 0.90 ms at 51 edges a node, 0.84 -> 0.87 at 200; 64 / 32 0.86 -> 0.89 there and 5.94 -> 6.00 at
    258.
    The summed backward takes rows of at most 1024 floats over all kernels, and keeps the kernels in registers up to 256 each;
    wider outputs gather the aggregate's gradient, which has no such limit on them."""
    row = (fout + 3) // 4 * 4
    if row > 256 or k * row > 1024 or (k * fin <= 64 and e >= 128 * n):
        return False
    if not input_grad:
        return k * fin >= 2 * row
    return k * fin >= 3 * row and n * fin * k * fout <= 20 * e * (k * fin - row)


def GmmAggregateLinear(rowptr, colind, colptr, rowind, permute, feat, pseudo, pseudo_csc, mu, sigma, weight, own_order=False, bias=None):
    """sum_k (sum_p w[p,k] * feat[colind[p],:]) @ W_k for feat [N, in] and the fc weight [K*out, in]: [N, out].  The forward aggregates the
    input (an edge gathers `in` floats); the backward takes the other order of the two linear steps, so an edge gathers the `out`
    floats of the gradient: T[j,k,:] = sum_p w[p,k] * g[row(p),:] is the gradient of feat @ W_k^T, the derivatives of the Gaussian weights
    need <g[row(p),:], (feat @ W_k^T)[j,:]>, and the projection is formed again.  With one copy of the coordinates nothing as wide as K x in
    is kept.
    pseudo_csc, own_order: as GmmConvFuseSumTwoOrders; pseudo_csc None: one copy, through permute.  bias [out]: added in the product's store
    (169 k x 64: the layer's forward and backward 985 -> 978 us)."""
    return GmmAggregateLinearFunction.apply(rowptr, colind, colptr, rowind, permute, feat, pseudo, pseudo_csc, mu, sigma, weight, own_order, bias)


def _matmul_in_parts(a, b, part):
    """a @ b, the inner dimension summed in parts.  The backward below takes the two linear steps in the other order, with the longer inner
    dimension in the product: as one chain its gradients of the coordinates and of the input were further from float64 than in the
    order of the forward (169 k nodes, 128 -> 64 with 3 kernels: 2.2e-7 against 1.7e-7; 300 k, 256 -> 128 with 4: 3.0e-7 and 4.1e-7 against
    2.3e-7 and 2.1e-7).  In parts of the layer's outputs they are as near (1.7e-7; 2.3e-7 and 2.1e-7), for a pass over the result
    per part: layer steps 1.01 -> 1.03 and 3.07 -> 3.24 ms."""
    part = max(32, part // 16 * 16)
    out = torch.matmul(a[:, :part], b[:part])
    for c in range(part, a.shape[1], part):
        out.addmm_(a[:, c:c + part], b[c:c + part])
    return out


class _AggregateHistory(torch.autograd.Function):
    """An aggregate that is there already, as the result of GmmAggregate / GmmAggregateTwoOrders: the value of `agg`, their backward."""

    @staticmethod
    def forward(ctx, agg, colptr, rowind, permute, feat, pseudo, mu, sigma, own_order):
        ctx.save_for_backward(colptr, rowind, permute, feat, pseudo, mu, sigma)
        ctx.own_order = own_order
        return agg.view_as(agg)

    @staticmethod
    def backward(ctx, grad_out):
        grads = gmm_native.gmmconv_shared_backward(*ctx.saved_tensors, grad_out.contiguous(), own_order=ctx.own_order)
        return (None, None, None, None) + grads + (None,)


class GmmAggregateLinearFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rowptr, colind, colptr, rowind, permute, feat, pseudo, pseudo_csc, mu, sigma, weight, own_order, bias=None):
        k, fin = mu.shape[0], feat.shape[1]
        fout = weight.shape[0] // k
        agg = gmm_native.gmmconv_shared(rowptr, colind, feat, pseudo, mu, sigma, own_order=own_order)
        w = weight.view(k, fout, fin).permute(1, 0, 2).reshape(fout, k * fin)
        ctx.two_orders, ctx.own_order = pseudo_csc is not None, own_order
        # for a graph of the gradients: the arrays to aggregate again, or, where the CSR copy of the coordinates is the caller's to reuse
        # after the forward, the aggregate
        ctx.save_for_backward(colptr, rowind, None if ctx.two_orders else permute, feat, pseudo_csc if ctx.two_orders else pseudo, mu, sigma, weight,
                              rowptr, colind, agg if ctx.two_orders else None)
        agg = agg.view(-1, k * fin)
        if product_wanted(agg, w, transposed=True, bias=bias):
            return tall_product(agg, w, transposed=True, bias=bias, asked=True)
        y = torch.matmul(agg, w.t())
        return y if bias is None else y + bias

    @staticmethod
    def backward(ctx, grad_out):
        from ..layers.dense import column_sum, reduce_over_rows
        colptr, rowind, permute, feat, pseudo, mu, sigma, weight, rowptr, colind, agg = ctx.saved_tensors
        k, fin = mu.shape[0], feat.shape[1]
        fout = weight.shape[0] // k
        grad_bias = column_sum(grad_out.contiguous()) if ctx.needs_input_grad[12] else None
        if torch.is_grad_enabled():
            # a graph of the gradients is wanted: the weight's gradient from the aggregate, by operations that record one, as in the
            # layer composed of GmmAggregate and a product (the other gradients come out of the library without history either way)
            if agg is None:
                agg = gmm_native.gmmconv_shared(rowptr, colind, feat, pseudo, mu, sigma, own_order=ctx.own_order)
            agg = _AggregateHistory.apply(agg.detach(), colptr, rowind, permute, feat, pseudo, mu, sigma, ctx.own_order).view(-1, k * fin)
            g = grad_out.contiguous()
            grad_w = reduce_over_rows(g, agg).view(fout, k, fin).permute(1, 0, 2).reshape(k * fout, fin)
            grad_agg = torch.matmul(g, weight.view(k, fout, fin).permute(1, 0, 2).reshape(fout, k * fin)).view(-1, k, fin)
            grad_feat, grad_pseudo, grad_mu, grad_sigma = gmm_native.gmmconv_shared_backward(colptr, rowind, permute, feat, pseudo, mu, sigma, grad_agg,
                                                                                             own_order=ctx.own_order)
            gp = (None, grad_pseudo) if ctx.two_orders else (grad_pseudo, None)
            return (None, None, None, None, None, grad_feat) + gp + (grad_mu, grad_sigma, grad_w, None, grad_bias)
        pad = (-fout) % 4
        if pad:         # zero columns up to a multiple of 4: the operator then takes its 128-bit row layout
            weight = torch.nn.functional.pad(weight.view(k, fout, fin), (0, 0, 0, pad)).view(-1, fin)
            grad_out = torch.nn.functional.pad(grad_out, (0, pad))
        proj = _matmul_in_parts(feat, weight.t(), fout).view(-1, k, fout + pad)
        t, grad_pseudo, grad_mu, grad_sigma = gmm_native.gmmconv_backward(colptr, rowind, permute, proj, pseudo, mu, sigma, grad_out.contiguous(),
                                                                          sum_kernels=True, own_order=ctx.own_order)
        t = t.view(-1, k * (fout + pad))
        grad_feat = _matmul_in_parts(t, weight, fout) if ctx.needs_input_grad[5] else None
        grad_w = reduce_over_rows(t, feat) if ctx.needs_input_grad[10] else None
        if pad and grad_w is not None:
            grad_w = grad_w.view(k, fout + pad, fin)[:, :fout].reshape(-1, fin)
        gp = (None, grad_pseudo) if ctx.two_orders else (grad_pseudo, None)
        return (None, None, None, None, None, grad_feat) + gp + (grad_mu, grad_sigma, grad_w, None, grad_bias)


class GmmFuseSumFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma, bias=None, residual=None):
        out = gmm_native.gmmconv(rowptr, colind, node_feat, pseudo, mu, sigma, sum_kernels=True, bias=bias, residual=residual)      # [N, F]
        ctx.save_for_backward(rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma)
        ctx.has_bias, ctx.has_res = bias is not None, residual is not None
        return out

    @staticmethod
    def backward(ctx, grad_out):
        rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma = ctx.saved_tensors
        grad_feat, grad_pseudo, grad_mu, grad_sigma = gmm_native.gmmconv_backward(
            colptr, rowind, permute, node_feat, pseudo, mu, sigma, grad_out.contiguous(), sum_kernels=True)
        return (None, None, None, None, None, grad_feat, grad_pseudo, grad_mu, grad_sigma) + _epilogue_grads(ctx, grad_out.contiguous(), 9)


def GmmConvFuseEb(rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma):
    return GmmFuseEbFunction.apply(rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma)


class GmmFuseEbFunction(GmmFuseFunction):
    """The reference's edge-balanced variant (operators/fused_gmmconv.py:61-79).  Load balance is
    handled by the degree-binned schedule here, so it is the same computation."""


def GaussianCp(pseudo, mu, sigma):
    return GaussianFunction.apply(pseudo, mu, sigma)


class GaussianFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, pseudo, mu, sigma):
        out = gmm_native.Gaussian(pseudo, mu, sigma)
        ctx.save_for_backward(pseudo, mu, sigma)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        pseudo, mu, sigma = ctx.saved_tensors
        return gmm_native.GaussianBp(pseudo, mu, sigma, grad_out.contiguous())


def GmmConvStash(rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma):
    return GmmStashFunction.apply(rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma)


class GmmStashFunction(torch.autograd.Function):
    """Stash variant (operators/fused_gmmconv.py:100-118): the forward also writes the Gaussian
    weights [E,K].  The backward uses the same single CSC pass as GmmFuseFunction (recomputing
    the weights is cheaper than reading them back through `permute`)."""

    @staticmethod
    def forward(ctx, rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, sigma):
        out, gauss = gmm_native.gmmconv(rowptr, colind, node_feat, pseudo, mu, sigma, want_gauss=True)
        ctx.save_for_backward(rowptr, colind, colptr, rowind, permute, gauss, node_feat, pseudo, mu, sigma)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        rowptr, colind, colptr, rowind, permute, gauss, node_feat, pseudo, mu, sigma = ctx.saved_tensors
        grad_feat, grad_pseudo, grad_mu, grad_sigma = gmm_native.gmmconv_backward(
            colptr, rowind, permute, node_feat, pseudo, mu, sigma, grad_out.contiguous())
        return None, None, None, None, None, grad_feat, grad_pseudo, grad_mu, grad_sigma
