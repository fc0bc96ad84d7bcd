"""Products over very many rows (one per node, point or edge) with a small matrix: csrc/fgnn_tall.hip."""
from __future__ import annotations

import torch

from .._lib import FgnnError, as_f32, check, device_guard, lib, ptr, stream_ptr, workspace


# Where a torch does not have the private names, its public mode stack is asked.
_modes = getattr(torch._C, "_len_torch_dispatch_stack", None) or (lambda: torch.utils._python_dispatch._get_current_dispatch_mode() is not None)
_transforms = getattr(torch._C, "_are_functorch_transforms_active", None) or (lambda: False)
_recording = getattr(torch._C, "_is_tracing", None) or torch.jit.is_tracing


def _traced():
    """Whether torch's own operations are being watched or rewritten (torch.compile, jit.trace, make_fx, fake tensors, functorch): a kernel launched past them
    would be missing from the record, or be handed no memory.  Asked before any size, so that no size becomes a condition of the record, and the
    compiler first: it does not follow the questions behind it."""
    return torch.compiler.is_compiling() or _recording() or bool(_modes()) or _transforms()


# These questions stand in front of every product, and small layers are bound by the host: each attribute is asked for once, and nothing twice (host time
# of the three rules and three wrappers of a layer with scores, launches left out: 65 us with generators over the operands and both asking, 39 so).
_TENSORS = (torch.Tensor, torch.nn.Parameter)


def _matrix(t):
    if not t.is_cuda or t.dtype is not torch.float32 or type(t) not in _TENSORS:
        return False
    strides = t.stride()
    if len(strides) != 2:
        return False
    columns = t.shape[1]
    return (strides[1] == 1 or columns == 1) and strides[0] >= columns


def _matrices(x, b=None):
    """fp32 matrices on one GPU with unit column stride (whatever torch calls the stride of a single column)."""
    return _matrix(x) and (b is None or (_matrix(b) and x.device == b.device))


def _plain(x, b=None):
    """Such matrices outside autocast (which asks for another precision)."""
    return not torch.is_autocast_enabled("cuda") and _matrices(x, b)


def _fits(shape, k, m, device, bias):
    """Whether x of `shape` on `device` has k columns and bias, where there is one, m floats beside it: the kernels read by these sizes alone."""
    return len(shape) == 2 and shape[1] == k and (bias is None or (bias.shape == (m,) and bias.dtype == torch.float32 and bias.device == device))


def product_wanted(x, b, *, transposed=False, bias=None, h_in=0, h_out=0, m=None):
    """Whether tall_product takes x [n, k] and the [k + 2 h_in, m + 2 h_out] matrix b (its transpose when `transposed`) and is the faster
    form; what does not fit goes to the library, which says so.  m: the columns, where b [k, .] is only what the matrix is laid out from.
    It reads x and writes the result once at 100-110 TFLOP/s, and every workgroup lays b out in LDS first, 5 to 30 us.  The library reaches 60-85
    TFLOP/s on thin shapes and more at the sizes it is tuned for, takes 19 us of the host at least (this kernel 11), and needs a score kernel (10 to
    600) or a stacked operand besides for extra columns.  The lines are drawn by the time of a call in a stream of calls, host included; us,
    library / own, in brackets of the GPU alone, as in a replayed graph, where that is another order.
    No extra columns.  Up to 49 k rows 4 k x 64 -> 64 21 / 12 (4.4 / 6.6), 16 k x 64 -> 128 20 / 12 (7.3 / 11.5), 33 k x 64 -> 128 21 / 15 (10.8 / 14.4),
    33 k x 256 -> 128 22 / 31.  Up to 131 k rows: 65 k x 16 -> 64 20 / 11, 64 -> 64 20 / 14 (11.4 / 13.8), 64 -> 128 20 / 23; 131,071 x 64 -> 64 22 / 22,
    64 -> 128 32 / 35.  Above: 140 k x 64 -> 128 47 / 37, 384 -> 64 85 / 78, 256 -> 128 94 / 100; 169 k x 64 -> 64 48 / 26, 64 -> 128 63 / 43, 128 -> 128
    87 / 68, 384 -> 64 171 / 97, 64 -> 256 72 / 77, 256 -> 128 108 / 121, 602 -> 48 122 / 138; 300 k x 128 -> 128 129 / 110, 602 -> 48 206 / 221; 700 k x
    64 -> 128 217 / 141, 602 -> 48 455 / 470; 1 M x 64 -> 256 423 / 360.  A power of two of the library's row tiles is what it is tuned for: 131 k x
    64 -> 64 22 / 22, 128 -> 64 29 / 32, 256 -> 64 44 / 53; 262 k x 64 -> 64 38 / 34, 64 -> 128 57 / 58, 128 -> 128 87 / 96; 524 k x 64 -> 128 114 / 113,
    128 -> 128 172 / 179 (a row less 172 / 181); 1 M x 128 -> 64 206 / 192, 256 -> 64 331 / 344.
    With them, scores included: 4 k x 64 -> 64 + 8 30 / 14, 256 -> 64 + 8 29 / 18 (8.6 / 17.3), 128 -> 256 + 8 29 / 28 (9.7 / 27.6); 16 k x 64 -> 64 + 8
    29 / 14, 256 -> 48 + 2 29 / 17 (14.5 / 16.9), 128 -> 256 + 8 29 / 33; 65 k 30 / 15, 35 / 29, 54 / 54; 169 k 60 / 33, 85 / 68, 142 / 138; 1 M 231 /
    137, 521 / 323, 761 / 601.  Gradients, stacking and the weights' included: 4 k x 64 + 8 -> 64 56 / 29; 49 k 48 + 2 -> 256 67 / 58, 256 + 8 -> 128 101 /
    109; 65,536 x 48 + 2 -> 256 66 / 65, 128 + 16 -> 128 76 / 79, 256 + 8 -> 128 129 / 123; a row more 85 / 79 (8 scores), 110 / 89, 158 / 136; 1 M x 64 + 8
    -> 64 401 / 142, 48 + 2 -> 256 628 / 348, 256 + 8 -> 128 1216 / 598 (these without the weights' gradient)."""
    if _traced():
        return False
    shape, rows = x.shape, b.shape
    if len(rows) != 2:
        return False
    k = rows[1 if transposed else 0] - 2 * h_in
    if m is None:
        m = rows[0 if transposed else 1] - 2 * h_out
    if not _fits(shape, k, m, x.device, bias):
        return False
    n = shape[0]
    if h_out or h_in:
        most = 73728 if n >= 65536 else 20480 if h_out else 16384
    elif n < 131072:
        most = 8192 if n <= 49152 else 4096
    else:
        tiles = -(-n // 256)
        most = (4096 if n <= 1 << 18 else 8192) if tiles & (tiles - 1) == 0 else 8192 if m > 192 and n < (1 << 19) else 24576
    return (n > 0 and k > 0 and m > 0 and max(h_in, h_out) <= 8 and (k + 2 * h_in) * (m + 2 * h_out) <= most
            and k <= 1024 and m <= 512 and _plain(x, b) and (not h_in or (k % 4 == 0 and x.data_ptr() % 16 == 0 and x.stride(0) % 4 == 0)))


def reduce_wanted(x, g, h=0):
    """Where tall_reduce of x [n, a] and g [n, b] (and 2h extra columns) is the faster form: one launch and a small sum for a batched product
    over chunks, a sum, the rows past the last chunk of 2048, and a stacked operand where there are extra columns (us, library / own, host included;
    in brackets of the GPU alone where that is another order).  On few rows the sum over the workgroups' results is what takes the time, so those are
    small ones there: 4 k x 64, 64 28 / 15, 64, 128 28 / 20, 128, 128 28 / 29; 33 k x 64, 128 28 / 21 (14 / 21), 128, 128 27 / 31.  Beyond: 52,001 x 128, 128
    57 / 33, 131,071 x 192, 128 85 / 72.  Whole chunks leave the library no remainder: 57 k x 128, 128 34 / 32, 65,536 x 64, 64 28 / 18 (15.4 / 17.5), 64, 128
    28 / 23, 128, 128 28 / 33, 122,880 x 64, 128 35 / 35, 128, 128 44 / 51, 131,072 x 64, 64 27 / 27, 64, 128 28 / 36.  Above 131 k rows either is as fast
    (233 k x 602, 32 228 / 242, 169 k x 384, 64 112 / 116).  With extra columns: 4 k x 64, 64 + 8 61 / 18, 65 k x 256, 48 + 2 62 / 35, 128, 256 + 8
    62 / 62; 169 k x 64, 64 + 8 69 / 40, 256, 48 + 2 100 / 73, 128, 256 + 8 229 / 135; 1 M 341 / 184, 444 / 375, 1153 / 684."""
    if _traced():
        return False
    xs, gs = x.shape, g.shape
    if len(xs) != 2 or len(gs) != 2 or xs[0] != gs[0]:
        return False
    n, a, b = xs[0], xs[1], gs[1]
    tiles = -(-a // 16) * (-(-b // 16) + (h > 0))
    whole = h == 0 and n >= 65536 and n % (n // 2048) == 0
    return (n > 0 and a > 0 and b > 0 and a + b <= 1024 and a % 4 == 0 and b % 4 == 0 and h <= 8 and tiles <= (36 if n <= 49152 or whole else 144)
            and (h > 0 or n < 131072) and _plain(x, g) and x.stride(0) % 4 == 0 and g.stride(0) % 4 == 0 and x.data_ptr() % 16 == 0 and g.data_ptr() % 16 == 0)


def _columns(x, extra):
    """Whether extra is None or two contiguous [n, h] arrays beside x [n, .]."""
    if extra is None:
        return True
    one, two = extra
    return (one.is_contiguous() and two.is_contiguous() and one.dtype is two.dtype is torch.float32 and one.device == x.device == two.device
            and one.shape == two.shape and len(one.shape) == 2 and one.shape[0] == x.shape[0])


def tall_product(x, b, *, transposed=False, bias=None, extra_in=None, extra_out=0, asked=False):
    """x [n, k] @ b (b^T when `transposed`) (+ bias).  extra_in: two [n, h] arrays that follow x's columns; extra_out: h, the last 2h
    columns of the result are returned as two [n, h] arrays of their own.  asked: product_wanted has just said so of these operands, which are not
    looked over again (b may be what the weights it saw were laid out in); extra_in are the gradients of two fp32 [n, h] outputs, made contiguous,
    whose shape and device autograd has seen to."""
    n, k = shape = x.shape
    rows = b.shape
    hin = 0 if extra_in is None else extra_in[0].shape[1]
    m = rows[0 if transposed else 1] - 2 * extra_out
    if not ((asked or (_matrices(x, b) and _fits(shape, k, m, x.device, bias) and _columns(x, extra_in))) and m >= 1
            and rows[1 if transposed else 0] == k + 2 * hin):
        raise FgnnError("tall_product: x %s, matrix %s%s, bias %s and %d + %d extra columns do not fit one another" % (
            tuple(x.shape), tuple(b.shape), " (transposed)" if transposed else "", None if bias is None else tuple(bias.shape), hin, extra_out))
    bias = None if bias is None else as_f32(bias)
    y = torch.empty((n, m), dtype=torch.float32, device=x.device)
    e0 = torch.empty((n, extra_out), dtype=torch.float32, device=x.device) if extra_out else None
    e1 = torch.empty_like(e0) if extra_out else None
    x0, x1 = extra_in if hin else (None, None)
    with device_guard(x.device):
        check(lib().fgnn_tall_product(n, k, m, ptr(x), x.stride(0), ptr(b), b.stride(0), int(transposed), ptr(bias), ptr(y), m, hin, ptr(x0), ptr(x1), extra_out,
                                      ptr(e0), ptr(e1), stream_ptr()), "fgnn_tall_product")
    return (y, e0, e1) if extra_out else y


def tall_reduce(x, g, extra=None, asked=False):
    """x [n, a]^T @ g [n, b] -> [a, b]; extra: two [n, h] arrays that follow g's columns; asked: of reduce_wanted, as above."""
    n, a = x.shape
    b = g.shape[1]
    h = 0 if extra is None else extra[0].shape[1]
    if not (asked or (_matrices(x, g) and g.shape[0] == n and _columns(x, extra))):
        raise FgnnError("tall_reduce: x %s, g %s and 2 x %d extra columns do not fit one another" % (tuple(x.shape), tuple(g.shape), h))
    c = torch.empty((a, b + 2 * h), dtype=torch.float32, device=x.device)
    e0, e1 = extra if h else (None, None)
    with device_guard(x.device):
        ws, wsb = workspace(lib().fgnn_tall_reduce_workspace_bytes(n, a, b, h), x.device)
        check(lib().fgnn_tall_reduce(n, a, b, ptr(x), x.stride(0), ptr(g), g.stride(0), h, ptr(e0), ptr(e1), ptr(c), ptr(ws), wsb, stream_ptr()), "fgnn_tall_reduce")
    return c


def sum_wanted(g):
    """Where tall_sum of g [n, c] is the faster form: two launches for torch's one or two, or five with columns that are no multiple of four (us,
    torch / own, host included: 33 k x 64 11 / 13, 66 k x 16 10 / 11, 169 k x 16 12 / 12, 64 20 / 13, 41 31 / 11, 1 23 / 20, of the GPU 10 / 20)."""
    return not _traced() and g.dim() == 2 and g.shape[0] >= 131072 and 3 <= g.shape[1] <= 1024 and _plain(g)


def tall_sum(g):
    """The column sums of g [n, c]."""
    n, c = g.shape
    if not _matrices(g):
        raise FgnnError("tall_sum: not an fp32 matrix on the GPU with unit column stride")
    out = torch.empty(c, dtype=torch.float32, device=g.device)
    with device_guard(g.device):
        ws, wsb = workspace(lib().fgnn_column_sum_workspace_bytes(n, c), g.device)
        check(lib().fgnn_column_sum(n, c, ptr(g), g.stride(0), ptr(out), ptr(ws), wsb, stream_ptr()), "fgnn_column_sum")
    return out
