"""Dense projections on MI355X: the library's own products (asrn_gemm) where they are the faster ones, and a weight
gradient that fits a long token axis.

For y = x W^T + b over N tokens, the weight gradient dW = dY^T X reduces over all N (32768 at the layer benchmark's
shape) into a small (out, in) matrix. As one GEMM it has only (out / tile) x (in / tile) output tiles to spread over
256 CUs. asrn_gemm cuts the token axis into slabs whose partial products are added in order, and sums the bias
gradient (dY's columns) from the values it loads anyway. fp32 products run there on the bf16 matrix cores, each operand
split into three bf16 parts: fp32's error (for operands from 2^-110 on) at more than fp32's matrix rate. Where hipBLASLt
is faster (below), it is called as before: the weight gradient as one batched product over slabs of tokens.
Under autocast the operands are cast as autocast casts F.linear's, and the products run in that dtype.

On the GPU, the sums (the slab partials, and the bias gradients' column sums) run in the library's asrn_column_sums
(fp32 accumulation in a fixed order, no memset-cleared semaphores, safe to capture in a HIP graph). fp64 operands,
and CPU tensors (the math checked on the CPU), use torch's sums.
"""
import math

import torch
import torch.nn.functional as F

from . import _lib

MIN_SLAB = 1024            # tokens per slab: below this the batched GEMM's own overhead dominates
MAX_SLAB_WEIGHT = 1 << 20  # weights with this many elements or more keep one GEMM: enough output tiles already, and
                           # S partial copies of them would cost more traffic than they save


def slabs_for(n, weight_elems=0):
    """Slab count for a token axis of n: 16 (or fewer) slabs of at least MIN_SLAB tokens that divide n exactly; 1 for
    weights of MAX_SLAB_WEIGHT elements or more."""
    if weight_elems >= MAX_SLAB_WEIGHT:
        return 1
    for s in (16, 8, 4, 2):
        if n % s == 0 and n // s >= MIN_SLAB:
            return s
    return 1


def _rows(t):
    """(N, k) view of a (..., k) tensor whose last axis is contiguous; copies only when the leading axes do not
    flatten to one stride."""
    k = t.shape[-1]
    n = math.prod(t.shape[:-1])                      # stated: -1 has no value for a zero-wide t
    if t.stride(-1) != 1:
        t = t.contiguous()
    try:
        return t.view(n, k)
    except RuntimeError:
        return t.reshape(n, k)


def _slab(t, s):
    """(s, N / s, k) view of an (N, k) matrix with unit last stride (splitting the row axis never needs a copy)."""
    n, k = t.shape
    return t.view(s, n // s, k)


# fp32 products of fewer multiply-adds than this stay on hipBLASLt, measured (us, it / asrn_gemm): 2048 x 64 x 256
# 5.9 / 9.1, 4611 x 384 x 192 10.7 / 11.3, 5005 x 256 x 512 19.1 / 17.8, 4611 x 384 x 384 17.6 / 16.0, 32768 x 256 x 256
# 39.1 / 33.1, 12000 x 768 x 3072 492 / 303: below, a launch's few steps wait for their loads
MIN_PRODUCTO = 400_000_000
# fp32 weight gradients over fewer tokens stay there too: 64 x 64 over 200 tokens 7.7 / 9.9, 64 x 256 over 2048 19.0 / 9.6
MIN_FICHAS = 512
# bf16 weight gradients on asrn_gemm: weights too large for slab copies (768 x 3072 over 16384 tokens 154 / 120,
# 1536 x 768 115 / 72) and small ones (112 x 128 12.4 / 11.4, 64 x 1024 over 65536 34 / 32, 512 x 256 over 5008
# 18.7 / 15.1); between them hipBLASLt's batched slabs win (768 x 768 35 / 51, 512 x 512 over 65536 55 / 69)
MAX_PESO_16 = 1 << 17
# Of the large ones, only over enough tokens for their partial products: tokens times this at least the weight's elements,
# with the bias gradient (13 us or more as a launch of its own) and without. 768 x 3072 with it over 2048 tokens 37 / 48,
# over 5001 68 / 63, 512 x 2048 over 3000 41 / 33, 8000 x 512 over 8192 105 / 111; without it 768 x 3072 over 8192 77 / 81,
# 1536 x 768 over 4097 35 / 39, over 8192 60 / 52, 32768 x 768 over 16384 763 / 1109
FICHAS_PESO = {True: 400, False: 200}


def _apto(t):
    """Whether asrn_gemm can read the 2-D matrix t in place."""
    return (t.dim() == 2 and t.stride(1) == 1 and t.stride(0) % 4 == 0 and t.stride(0) >= t.shape[1]
            and t.data_ptr() % (4 * t.element_size()) == 0)


def gemm(a, ta, b, tb, sesgo=None, columnas=False):
    """op(a) op(b) (+ sesgo) in fp32 on asrn_gemm, op the transpose where ta, tb. columnas (ta): returns (product, the
    sums of a's columns). Shapes that do not chain are refused here: the kernels see leading dimensions only and would
    read whatever lies there."""
    M, K = (a.shape[1], a.shape[0]) if ta else a.shape
    Kb, N = (b.shape[1], b.shape[0]) if tb else b.shape
    if K != Kb or (sesgo is not None and tuple(sesgo.shape) != (N,)):
        raise ValueError(f'gemm: shapes {tuple(a.shape)}{" transposed" if ta else ""}, {tuple(b.shape)}'
                         f'{" transposed" if tb else ""} and bias {None if sesgo is None else tuple(sesgo.shape)} do not chain')
    bf = int(a.dtype == torch.bfloat16)
    out = torch.empty((M, N), dtype=torch.float32, device=a.device)
    cols = torch.empty((M,), dtype=torch.float32, device=a.device) if columnas else None
    wsb = _lib.query('asrn_gemm_workspace', M, N, K, bf, int(columnas), 0, 0)
    ws = torch.empty((wsb,), dtype=torch.uint8, device=a.device) if wsb > 0 else None
    _lib.call('asrn_gemm', _lib.ptr(a), a.stride(0), int(ta), _lib.ptr(b), b.stride(0), int(tb), bf, _lib.ptr(out),
              out.stride(0), M, N, K, _lib.ptr(sesgo), 0, _lib.ptr(cols), 0, 0, _lib.ptr(ws), wsb,
              _lib.stream_of(a.device))
    return (out, cols) if columnas else out


def gemm_ok(a, b, tb, sesgo=None):
    """Whether a @ op(b) (+ sesgo) runs on asrn_gemm: fp32 on the GPU, aligned, MIN_PRODUCTO multiply-adds or more, and
    shapes that chain with one bias value per column (F.linear broadcasts a bias or refuses the rest)."""
    if b.dim() != 2 or a.shape[1] != b.shape[1 if tb else 0]:
        return False
    (M, K), N = a.shape, b.shape[0 if tb else 1]
    return (a.is_cuda and a.dtype == b.dtype == torch.float32 and b.device == a.device and M * N * K >= MIN_PRODUCTO
            and max(M, N, K) < 1 << 30 and N >= 64 and N % 4 == 0 and K % 4 == 0 and _apto(a) and _apto(b)
            and (sesgo is None or (sesgo.dtype == torch.float32 and sesgo.device == a.device and tuple(sesgo.shape) == (N,)
                                   and sesgo.is_contiguous() and sesgo.data_ptr() % 16 == 0)))


def _gradiente_ok(g2, x2, sesgo):
    """Whether dW = g2^T x2 runs on asrn_gemm (see the constants above)."""
    if not (g2.is_cuda and g2.dtype == x2.dtype and g2.dtype in (torch.float32, torch.bfloat16) and _apto(g2)
            and _apto(x2) and g2.shape[1] % 4 == 0 and x2.shape[1] % 4 == 0 and 1 <= g2.shape[0] < 1 << 30):
        return False
    n, peso = g2.shape[0], g2.shape[1] * x2.shape[1]
    if peso == 0:                      # no product to form, but the bias gradient still is (asrn_gemm returns at once)
        return False
    if g2.dtype == torch.float32:
        return sesgo or n >= MIN_FICHAS
    if peso >= MAX_SLAB_WEIGHT:
        return n * FICHAS_PESO[sesgo] >= peso
    return peso <= MAX_PESO_16 or slabs_for(n, peso) == 1


def _acc_dtype(t):
    return torch.float64 if t.dtype == torch.float64 else torch.float32


def _hip_sums(x, rows, cols, ld):
    """fp32 column sums of the (rows, cols) matrix at x (row stride ld) through asrn_column_sums."""
    out = torch.empty((cols,), dtype=torch.float32, device=x.device)
    wsb = _lib.query('asrn_column_sums_workspace', rows, cols)
    ws = torch.empty((wsb,), dtype=torch.uint8, device=x.device) if wsb > 0 else None
    _lib.call('asrn_column_sums', _lib.ptr(x), int(x.dtype == torch.bfloat16), rows, cols, ld, _lib.ptr(out),
              _lib.ptr(ws), wsb, _lib.stream_of(x.device))
    return out


def _on_hip(t):
    return t.is_cuda and t.dtype in (torch.float32, torch.bfloat16)


def sum_rows(t):
    """t (S, ...) summed over its first axis in fp32 (fp64 for fp64), in order."""
    if _on_hip(t):
        t = t.contiguous()
        n = t[0].numel() if t.shape[0] else 0
        return _hip_sums(t, t.shape[0], n, max(n, 1)).view(t.shape[1:])
    return t.sum(0, dtype=_acc_dtype(t))


def weight_grad(g2, x2, sesgo=False):
    """dW = g2^T x2, summed in fp32 (fp64 for fp64 operands): g2 (N, out), x2 (N, in), both with unit last stride.
    sesgo: (dW, the bias gradient column_sums(g2))."""
    if _gradiente_ok(g2, x2, sesgo):
        return gemm(g2, True, x2, False, columnas=sesgo)
    if sesgo:
        return weight_grad(g2, x2), column_sums(g2)
    s = slabs_for(g2.shape[0], g2.shape[1] * x2.shape[1])
    if s == 1:
        return g2.t().mm(x2).to(_acc_dtype(g2))
    # left operand: the transposed slab of g2; right operand: x2's slab as stored (never a transposed view)
    return sum_rows(torch.bmm(_slab(g2, s).transpose(1, 2), _slab(x2, s)))


def column_sums(g2):
    """Sum over the rows of g2 (N, k) with unit last stride, in fp32 (fp64 for fp64)."""
    if _on_hip(g2):
        return _hip_sums(g2, g2.shape[0], g2.shape[1], max(g2.stride(0), g2.shape[1], 1))
    return g2.sum(0, dtype=_acc_dtype(g2))


class _Lineal(torch.autograd.Function):

    @staticmethod
    def forward(ctx, x, w, b, dt, propio):
        xc, wc = x.to(dt), w.to(dt)
        bc = b.to(dt) if b is not None else None
        # rows flattened (which may copy) only for products that asrn_gemm takes by their size
        x2 = None
        if propio and xc.is_cuda and xc.dtype == torch.float32 and xc.numel() * wc.shape[0] >= MIN_PRODUCTO:
            x2 = _rows(xc)
        if x2 is not None and gemm_ok(x2, wc, True, bc):
            y = gemm(x2, False, wc, True, sesgo=bc).view(*x.shape[:-1], wc.shape[0])
        else:
            with torch.autocast(device_type=x.device.type, enabled=False):
                y = F.linear(xc, wc, bc)
        ctx.save_for_backward(xc, wc)
        ctx.meta = (x.dtype, w.dtype, None if b is None else b.dtype)
        return y

    @staticmethod
    def backward(ctx, g):
        xc, wc = ctx.saved_tensors
        xdt, wdt, bdt = ctx.meta
        gx = gw = gb = None
        with torch.autocast(device_type=g.device.type, enabled=False):
            g = g.to(wc.dtype)
            g2 = _rows(g)
            if ctx.needs_input_grad[0]:
                if gemm_ok(g2, wc, False):
                    gx = gemm(g2, False, wc, False).view(*g.shape[:-1], wc.shape[1]).to(xdt)
                else:
                    gx = g.matmul(wc).to(xdt)
            con_sesgo = bdt is not None and ctx.needs_input_grad[2]
            if ctx.needs_input_grad[1]:
                gw = weight_grad(g2, _rows(xc), con_sesgo)
                if con_sesgo:
                    gw, gb = gw[0], gw[1].to(bdt)
                gw = gw.to(wdt)
            elif con_sesgo:
                gb = column_sums(g2).to(bdt)
        return gx, gw, gb, None, None


def lineal(x, w, b=None, propio=True):
    """F.linear(x, w, b) with its products on asrn_gemm where that is faster; honours autocast like F.linear.
    propio=False: the forward stays F.linear's (outputs whose signs are hashed keep its rounding)."""
    dev = x.device.type
    dt = torch.get_autocast_dtype(dev) if torch.is_autocast_enabled(dev) else x.dtype
    return _Lineal.apply(x, w, b, dt, propio)
