"""GMMConv (MoNet) layers on the fused operators (interface of the reference's
layers/gmmconv_layer.py:17-76 and :221-282)."""
from __future__ import annotations

import torch as th
from torch import nn
from torch.nn import init

from .._lib import xcd_buckets_enabled
from ..operators.edge_proj import edge_linear_tanh
from ..operators.fused_gmmconv import (GmmAggregate, GmmAggregateLinear, GmmAggregateTwoOrders, GmmConvFuseSum, GmmConvFuseSumTwoOrders, GmmConvStash,
                                        GmmConvStashSumTwoOrders, GmmProjectedTwoOrders, gmm_native, project_in_backward, projected_pays)
from .dense import add_bias, tall_linear


class _GMMBase(nn.Module):
    _op = None          # callable(rowptr, colind, colptr, rowind, permute, node_feat, pseudo, mu, inv_sigma) -> [N, F]

    def __init__(self, in_feats, out_feats, dim, n_kernels, aggregator_type="sum", residual=False, bias=True,
                 allow_zero_in_degree=False):
        super().__init__()
        if aggregator_type != "sum":
            raise KeyError("Aggregator type {} not recognized.".format(aggregator_type))
        self._out_feats = out_feats
        self._dim = dim
        self._n_kernels = n_kernels
        self._allow_zero_in_degree = allow_zero_in_degree
        self.mu = nn.Parameter(th.empty(n_kernels, dim))
        self.inv_sigma = nn.Parameter(th.empty(n_kernels, dim))
        self.fc = nn.Linear(in_feats, n_kernels * out_feats, bias=False)
        if residual:
            self.res_fc = nn.Linear(in_feats, out_feats, bias=False) if in_feats != out_feats else nn.Identity()
        else:
            self.register_buffer("res_fc", None)
        if bias:
            self.bias = nn.Parameter(th.empty(out_feats))
        else:
            self.register_buffer("bias", None)
        self.reset_parameters()

    def reset_parameters(self):
        # layers/gmmconv_layer.py:55-62: Xavier-normal fc, mu ~ N(0, 0.1), inv_sigma = 1, bias = 0
        gain = init.calculate_gain("relu")
        init.xavier_normal_(self.fc.weight, gain=gain)
        if isinstance(self.res_fc, nn.Linear):
            init.xavier_normal_(self.res_fc.weight, gain=gain)
        init.normal_(self.mu.data, 0, 0.1)
        init.constant_(self.inv_sigma.data, 1)
        if self.bias is not None:
            init.zeros_(self.bias.data)

    def set_allow_zero_in_degree(self, set_value):
        self._allow_zero_in_degree = set_value

    def forward(self, rowptr, colind, colptr, rowind, permute, feat, pseudo, pseudo_csc=None, own_order=False, proj=None):
        """pseudo_csc: the same pseudo-coordinates in CSC order, pseudo[permute], built by
        the caller from its own CSC-ordered edge data.  The backward then works in CSC order throughout
        and the gradient of the pseudo-coordinates flows through pseudo_csc instead of pseudo.
        own_order: pseudo and pseudo_csc are in the entry order of the operators' schedules
        (operators.fused_gmmconv.gmm_edge_positions); without pseudo_csc the layer is forward-only.
        proj: a Linear(2, dim) whose tanh gives the coordinates; pseudo and pseudo_csc are then raw [E, 2] pairs (constant data), and where the
        operators can, they project them on the way."""
        if proj is not None and not self._projects(feat, pseudo, pseudo_csc, proj, colptr, colind):
            apply = lambda t: edge_linear_tanh(t, proj.weight, proj.bias)
            if pseudo_csc is not None:
                with th.no_grad():
                    pseudo = apply(pseudo)
                pseudo_csc = apply(pseudo_csc)
            else:
                pseudo = apply(pseudo)
            proj = None
        if self._aggregate_first(feat):
            # without a residual the bias is added in the store of the product behind the aggregation (autocast and other types: as a sum of
            # its own, whose type is the wider one)
            bias = self.bias
            if bias is not None and (self.res_fc is not None or bias.dtype != th.float32 or th.is_autocast_enabled("cuda")):
                bias = None
            rst = self._forward_aggregate_first(rowptr, colind, colptr, rowind, permute, feat, pseudo, pseudo_csc, own_order, proj, bias)
            return rst if bias is not None else self._finish(rst, feat)
        node_feat = tall_linear(feat, self.fc.weight).view(-1, self._n_kernels, self._out_feats)    # = self.fc(feat)
        pad = (-self._out_feats) % 4
        if pad:         # zero columns up to a multiple of 4: the operator then takes its 128-bit row layout
            node_feat = th.nn.functional.pad(node_feat, (0, pad))
        # residual and bias (layers/gmmconv_layer.py:69-75 of the reference) go into the operator's store when the
        # width needs no padding; otherwise they are added afterwards
        fuse_tail = pad == 0 and (self.bias is not None or self.res_fc is not None)
        tail = lambda: {"bias": self.bias, "residual": None if self.res_fc is None else self.res_fc(feat)} if fuse_tail else {}
        if pseudo_csc is not None or own_order:
            if own_order and pseudo_csc is None and th.is_grad_enabled() and (node_feat.requires_grad or pseudo.requires_grad):
                raise ValueError("own_order without pseudo_csc is forward-only")
            if proj is not None:
                t = tail()
                rst = GmmProjectedTwoOrders(rowptr, colind, colptr, rowind, node_feat, pseudo, pseudo_csc, proj.weight, proj.bias, self.mu, self.inv_sigma,
                                            own_order, type(self)._op is not GmmConvFuseSum, t.get("bias"), t.get("residual"))
                return rst if fuse_tail else self._finish(rst[..., :self._out_feats], feat)
            two_orders = GmmConvFuseSumTwoOrders if (type(self)._op is GmmConvFuseSum or pseudo_csc is None) else GmmConvStashSumTwoOrders
            rst = two_orders(rowptr, colind, colptr, rowind, node_feat, pseudo.detach(), pseudo_csc, self.mu, self.inv_sigma,
                             own_order=own_order, **tail())
        elif type(self)._op is GmmConvFuseSum:
            rst = GmmConvFuseSum(rowptr, colind, colptr, rowind, permute, node_feat, pseudo, self.mu, self.inv_sigma, **tail())
        else:
            rst = type(self)._op(rowptr, colind, colptr, rowind, permute, node_feat, pseudo, self.mu, self.inv_sigma)
            fuse_tail = False
        if fuse_tail:
            return rst
        if pad:
            rst = rst[..., :self._out_feats]
        return self._finish(rst, feat)

    def _projects(self, feat, raw, raw_csc, proj, colptr, colind):
        """Whether this call leaves the projection to the operators: two orders of constant fp32 pairs, few kernels and coordinates, not the form
        of the layer whose backward takes the coordinates' gradient through a projection of the input, and edges enough to pay."""
        k, fin, n, e = self._n_kernels, feat.shape[1], feat.shape[0], colind.numel()
        if (raw_csc is None or not gmm_native.projection_supported(k, self._dim) or raw.requires_grad or raw_csc.requires_grad
                or any(t.dtype != th.float32 or not t.is_cuda for t in (raw, raw_csc, proj.weight, proj.bias))):
            return False
        first = self._aggregate_first(feat)
        if first and project_in_backward(k, fin, self._out_feats, feat.requires_grad, n, e):
            return False
        row = k * fin if first else (self._out_feats + 3) // 4 * 4
        return projected_pays(n, e, k, self._dim, row, first, xcd_buckets_enabled(colptr, e))

    def _finish(self, rst, feat):
        if self.res_fc is not None:
            rst = rst + self.res_fc(feat)
        if self.bias is not None:
            rst = add_bias(rst, self.bias)
        return rst

    def _aggregate_first(self, feat):
        """Whether the layer aggregates its input before the fc (recomputing layer only): when the input is
        narrower than the K x out floats an edge would gather otherwise, and the operator takes the shape."""
        k, fin = self._n_kernels, feat.shape[1]
        return (type(self)._op is GmmConvFuseSum and feat.dim() == 2 and fin < k * self._out_feats
                and gmm_native.shared_supported(k, fin))

    def _forward_aggregate_first(self, rowptr, colind, colptr, rowind, permute, feat, pseudo, pseudo_csc, own_order, proj=None, bias=None):
        """sum_k (sum_p w[p,k] feat[col(p),:]) @ W_k (+ bias): the reference's sum over k of the aggregated fc(feat)[:,k,:]
        (layers/gmmconv_layer.py:67-69) with the two linear steps exchanged."""
        k, fin, fout = self._n_kernels, feat.shape[1], self._out_feats
        feat = feat.contiguous()
        if pseudo_csc is not None or own_order:
            if own_order and pseudo_csc is None and th.is_grad_enabled() and (feat.requires_grad or pseudo.requires_grad):
                raise ValueError("own_order without pseudo_csc is forward-only")
        two = pseudo_csc is not None
        w = lambda: self.fc.weight.view(k, fout, fin).permute(1, 0, 2).reshape(fout, k * fin)       # [out, K*in]: rst = agg.view(N, K*in) @ w^T
        if proj is not None:
            agg = GmmProjectedTwoOrders(rowptr, colind, colptr, rowind, feat, pseudo, pseudo_csc, proj.weight, proj.bias, self.mu, self.inv_sigma, own_order)
            return tall_linear(agg.view(-1, k * fin), w(), bias)
        # without a gradient for what is aggregated (frozen Gaussians, constant coordinates and input) the weight's is one product with the
        # aggregate, and no pass over the edges
        through_edges = any(t.requires_grad for t in (feat, pseudo_csc if two else pseudo, self.mu, self.inv_sigma))
        if (th.is_grad_enabled() and through_edges and (two or not own_order)
                and project_in_backward(k, fin, fout, feat.requires_grad, feat.shape[0], colind.numel())):
            return GmmAggregateLinear(rowptr, colind, colptr, rowind, None if two else permute, feat, pseudo.detach() if two else pseudo, pseudo_csc,
                                      self.mu, self.inv_sigma, self.fc.weight, own_order=own_order, bias=bias)
        if two or own_order:
            agg = GmmAggregateTwoOrders(rowptr, colind, colptr, rowind, feat, pseudo.detach(), pseudo_csc, self.mu, self.inv_sigma,
                                        own_order=own_order)
        else:
            agg = GmmAggregate(rowptr, colind, colptr, rowind, permute, feat, pseudo, self.mu, self.inv_sigma)
        return tall_linear(agg.view(-1, k * fin), w(), bias)


class GMMConv(_GMMBase):
    """The `.sum(1)` over the mixture kernels of the reference layer (layers/gmmconv_layer.py:69) is
    fused into the operator."""
    _op = staticmethod(GmmConvFuseSum)


def _stash_sum(*args):
    return GmmConvStash(*args).sum(1)


class GMMConv_stash(_GMMBase):
    _op = staticmethod(_stash_sum)
