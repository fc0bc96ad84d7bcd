"""Products over very many rows (one per node, point or edge) with a small matrix: csrc/fgnn_tall.hip."""
from __future__ import annotations

import torch

from .._lib import as_f32, check, device_guard, lib, ptr, stream_ptr, workspace


def _plain(*ts):
    """fp32 matrices on one GPU with unit column stride, outside autocast (which asks for another precision)."""
    return all(t.is_cuda and t.dtype == torch.float32 and t.dim() == 2 and t.stride(1) == 1 and t.stride(0) >= t.shape[1] for t in ts) \
        and all(t.device == ts[0].device for t in ts) and not torch.is_autocast_enabled("cuda") and not torch.compiler.is_compiling()


def product_wanted(x, b, k, m, h_in=0, h_out=0):
    """Where tall_product of x [n, k] with the [k + 2 h_in, m + 2 h_out] matrix b is the faster form (us, library / own).  It reads x and
    writes the result once at 100-110 TFLOP/s; the library's products take 19 at least and reach 60-85 TFLOP/s on thin shapes, 150 on large
    ones.  Up to 8192 weights: 4 k rows x 64 -> 64 20 / 9, 33 k x 64 -> 128 19 / 14, 170 k 62 / 44; beyond that on many rows
    only (65 k x 64 -> 192 25 / 30, 128 -> 128 26 / 36; 170 k x 384 -> 64 181 / 108, 500 k x 128 -> 128 213 / 171), with more than 192
    columns on more still (170 k x 64 -> 256 72 / 83, 1 M 423 / 360).  With extra columns the library needs a score kernel (10 to 600) or a
    stacked operand besides: 8 k x 128 -> 144 20 + 10 / 17, 233 k x 256 -> 272 334 + 70 / 355, 2.4 M x 100 -> 272 1474 + 260 / 1310; 20 k rows of
    gradients 272 -> 256 33 + 8 / 53, 2.4 M 50 -> 256 1030 + 250 / 840."""
    n = x.shape[0]
    if h_out or (h_in and n >= 65536):
        most = 73728
    elif h_in:
        most = 16384
    else:
        most = 8192 if n < 131072 or (m > 192 and n < (1 << 19)) else 32768
    return (n > 0 and k > 0 and m > 0 and max(h_in, h_out) <= 8 and (k + 2 * h_in) * (m + 2 * h_out) <= most
            and k <= 1024 and m <= 512 and _plain(x, b) and (not h_in or (k % 4 == 0 and x.data_ptr() % 16 == 0 and x.stride(0) % 4 == 0)))


def reduce_wanted(x, g, h=0):
    """Where tall_reduce of x [n, a] and g [n, b] (and 2h extra columns) is the faster form: one launch and a small sum for a batched product
    over chunks, a sum, a remainder, and a stacked operand where there are extra columns (us, library / own: 33 k x 64, 128 32 / 23; 169 k x
    256, 42 98 + 30 / 80; 2.4 M x 256, 50 880 + 250 / 960; without extra columns, 233 k x 602, 32 228 / 242, 169 k x 384, 64 112 / 116)."""
    n, a, b = x.shape[0], x.shape[1], g.shape[1]
    tiles = -(-a // 16) * (-(-b // 16) + (h > 0))
    return (n > 0 and 0 < a + b <= 1024 and a > 0 and b > 0 and h <= 8 and tiles <= 144 and (h > 0 or n <= 131072) and _plain(x, g)
            and all(t.shape[1] % 4 == 0 and t.stride(0) % 4 == 0 and t.data_ptr() % 16 == 0 for t in (x, g)))


def tall_product(x, b, *, transposed=False, bias=None, extra_in=None, extra_out=0):
    """x [n, k] @ b (b^T when `transposed`) (+ bias).  extra_in: two [n, h] arrays that follow x's columns; extra_out: h, the last 2h
    columns of the result are returned as two [n, h] arrays of their own."""
    n, k = x.shape
    bias = None if bias is None else as_f32(bias)
    hin = 0 if extra_in is None else extra_in[0].shape[1]
    m = b.shape[0 if transposed else 1] - 2 * extra_out
    y = torch.empty((n, m), dtype=torch.float32, device=x.device)
    e0 = torch.empty((n, extra_out), dtype=torch.float32, device=x.device) if extra_out else None
    e1 = torch.empty_like(e0) if extra_out else None
    x0, x1 = extra_in if hin else (None, None)
    with device_guard(x.device):
        check(lib().fgnn_tall_product(n, k, m, ptr(x), x.stride(0), ptr(b), b.stride(0), int(transposed), ptr(bias), ptr(y), m, hin, ptr(x0), ptr(x1), extra_out,
                                      ptr(e0), ptr(e1), stream_ptr()), "fgnn_tall_product")
    return (y, e0, e1) if extra_out else y


def tall_reduce(x, g, extra=None):
    """x [n, a]^T @ g [n, b] -> [a, b]; extra: two [n, h] arrays that follow g's columns."""
    n, a = x.shape
    b = g.shape[1]
    h = 0 if extra is None else extra[0].shape[1]
    c = torch.empty((a, b + 2 * h), dtype=torch.float32, device=x.device)
    e0, e1 = extra if h else (None, None)
    with device_guard(x.device):
        ws, wsb = workspace(lib().fgnn_tall_reduce_workspace_bytes(n, a, b, h), x.device)
        check(lib().fgnn_tall_reduce(n, a, b, ptr(x), x.stride(0), ptr(g), g.stride(0), h, ptr(e0), ptr(e1), ptr(c), ptr(ws), wsb, stream_ptr()), "fgnn_tall_reduce")
    return c
