"""The Mamba block's token projections (in_proj, out_proj, prob_head of
e_model.py:258-506; in_prob of lra_impl.py:1490-1510) and their gradients.

fp32 products on the GPU run on this package's kernel (bcm_gemm_f32: the
operands split into two scaled fp16 values each, three products on the fp16
matrix cores, fp32 sums), which keeps fp32 accuracy (error against 64 bits
0.3 to 1 of the library's over the block's shapes) at up to 2.5 times the fp32
matrix cores' rate. One layer at 51 200 tokens, d_model 256, d_inner 512,
hipBLASLt before and here (us): in_proj 115 / 70, its input gradient 131 / 67,
its weight gradient 145 / 61; out_proj 152 / 65, its weight gradient 102 / 60;
prob_head's products 63 / 39.

A weight gradient reduces over every token of the batch: dW = dY^T X with a
small [out, in] result. The kernel splits the tokens over the chip and adds
the partials in a fixed order. Elsewhere (CPU, 16-bit, an open graph for a
second derivative) a product of at least 8192 tokens is split into 8 chunks,
one batched product and a fixed-order sum.
"""
import torch
import torch.nn.functional as F

try:
    from . import _native as _nat
except ImportError:  # imported with this directory on sys.path
    import _native as _nat

__all__ = ["linear", "mm", "proj_tokens_last", "weight_grad"]

SPLIT = 8
MIN_TOKENS = 8192


_PLAIN = (torch.Tensor, torch.nn.Parameter)
_LIMIT = 2 ** 31  # bytes: the kernel's 32-bit offsets


def _major(t, rows, cols):
    """(contiguous along dim 1, leading stride) of a 2-D operand whose rows
    or columns lie contiguous and apart, or None."""
    if t.stride(1) == 1 and (t.stride(0) >= cols or rows == 1):
        return True, max(t.stride(0), cols)
    if t.stride(0) == 1 and (t.stride(1) >= rows or cols == 1):
        return False, max(t.stride(1), rows)
    return None


def _kernel_form(x, y, bias=None):
    """The kernel's operand forms for x @ y (+ bias), or None where the
    product stays with torch: other types and devices, a product that
    autograd must see (no custom backward around it), autocast, a traced,
    wrapped or batched tensor, strides without a contiguous dimension, an operand of 2 GiB."""
    grad = torch.is_grad_enabled()
    for t in (x, y) if bias is None else (x, y, bias):
        if (type(t) not in _PLAIN or t.dtype != torch.float32 or not t.is_cuda or t.device != x.device
                or (grad and t.requires_grad) or _nat.no_memory(t)):
            return None
    if torch.is_autocast_enabled("cuda") or torch.compiler.is_compiling():
        return None
    if x.dim() != 2 or y.dim() != 2 or x.size(1) != y.size(0):
        return None
    (M, K), N = x.shape, y.size(1)
    if M == 0 or N == 0 or K == 0:
        return None
    if bias is not None and (bias.dim() != 1 or bias.size(0) != N or bias.stride(0) != 1):
        return None
    fx, fy = _major(x, M, K), _major(y, K, N)
    if fx is None or fy is None:
        return None
    (x_k, ldx), (y_n, ldy) = fx, fy
    if not x_k and not y_n:  # the one pair of layouts the kernel has no form for
        return None
    if ((M if x_k else K) + 128) * ldx * 4 >= _LIMIT or ((K if y_n else N) + 128) * ldy * 4 >= _LIMIT \
            or (M + 128) * N * 4 >= _LIMIT:
        return None
    return x_k, ldx, not y_n, ldy


def mm(x, y, bias=None):
    """x @ y (+ bias per column) of 2-D tensors."""
    form = _kernel_form(x, y, bias)
    if form is None:
        return x @ y if bias is None else torch.addmm(bias, x, y)
    return _kernel_mm(x, y, bias, form)


def _kernel_mm(x, y, bias, form):
    x_k, ldx, y_k, ldy = form
    (M, K), N = x.shape, y.size(1)
    out = torch.empty((M, N), dtype=torch.float32, device=x.device)
    with _nat.on_device(x.device):
        nbytes = 0 if bias is not None else int(_nat.lib().bcm_gemm_f32_workspace_bytes(M, N, K))
        ws = torch.empty(nbytes // 4, dtype=torch.float32, device=x.device) if nbytes else None
        _nat.call("bcm_gemm_f32", x.data_ptr(), int(x_k), ldx, y.data_ptr(), int(y_k), ldy,
                  bias.data_ptr() if bias is not None else None, M, N, K, out.data_ptr(), N, _nat.ptr(ws), nbytes,
                  _nat.stream_of(x))
    return out


def _split_ok(m, *ts):
    return m >= MIN_TOKENS and m % SPLIT == 0 and all(t.dtype == torch.float32 for t in ts)


def weight_grad(g, x, tokens_first=True):
    """Σ over tokens of g ⊗ x: gᵀ @ x for g [M, N] (tokens_first) or g @ x
    for g [N, M], with x [M, K]."""
    gt = g.t() if tokens_first else g
    form = _kernel_form(gt, x)
    if form is not None:
        return _kernel_mm(gt, x, None, form)
    m = x.size(0)
    if not _split_ok(m, g, x):
        return gt @ x
    c = m // SPLIT
    if tokens_first:
        gs = g.reshape(SPLIT, c, g.size(1)).transpose(1, 2)  # [S, N, c]
    else:
        gs = g.reshape(g.size(0), SPLIT, c).transpose(0, 1)  # [S, N, c]
    return torch.bmm(gs, x.reshape(SPLIT, c, x.size(1))).sum(0)


def column_sum(g):
    """g.sum(0) of a 2-D g: the bias gradient of a projection."""
    if (type(g) in _PLAIN and g.dtype == torch.float32 and g.is_cuda and 0 < g.numel() < _LIMIT
            and 4 <= g.size(1) <= 1024 and g.size(1) % 4 == 0 and g.is_contiguous()
            and not _nat.no_memory(g) and g.data_ptr() % 16 == 0
            and not (torch.is_grad_enabled() and g.requires_grad) and not torch.compiler.is_compiling()):
        rows, D = g.shape
        out = torch.empty(D, dtype=g.dtype, device=g.device)
        with _nat.on_device(g.device):
            nbytes = int(_nat.lib().bcm_column_sums_workspace_bytes(rows, D))
            ws = torch.empty(nbytes // 4, dtype=torch.float32, device=g.device)
            _nat.call("bcm_column_sums", g.data_ptr(), rows, D, out.data_ptr(), ws.data_ptr(), nbytes,
                      _nat.stream_of(g))
        return out
    return g.sum(0)


class _LinearFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias):
        ctx.save_for_backward(x, weight)
        ctx.has_bias = bias is not None
        if x.dim() > 1 and x.is_contiguous():
            x2, wt = x.view(-1, x.size(-1)) if x.numel() else x, weight.t()
            form = _kernel_form(x2, wt, bias)
            if form is not None:
                return _kernel_mm(x2, wt, bias, form).view(*x.shape[:-1], weight.size(0))
        return F.linear(x, weight, bias)

    @staticmethod
    def backward(ctx, gy):
        x, weight = ctx.saved_tensors
        g2 = gy.reshape(-1, gy.size(-1))
        dx = mm(g2, weight).view(x.shape) if ctx.needs_input_grad[0] else None
        dw = weight_grad(g2, x.reshape(-1, x.size(-1))) if ctx.needs_input_grad[1] else None
        db = column_sum(g2) if ctx.has_bias and ctx.needs_input_grad[2] else None
        return dx, dw, db


def linear(x, weight, bias=None):
    """F.linear(x, weight, bias) with this module's products."""
    return _LinearFn.apply(x, weight, bias)


class _ProjTokensLastFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, weight, h2d):
        ctx.save_for_backward(weight, h2d)
        return mm(weight, h2d.t())

    @staticmethod
    def backward(ctx, g):
        weight, h2d = ctx.saved_tensors
        dw = weight_grad(g, h2d, tokens_first=False) if ctx.needs_input_grad[0] else None
        dh = mm(g.t(), weight) if ctx.needs_input_grad[1] else None
        return dw, dh


def proj_tokens_last(weight, h2d):
    """weight @ h2dᵀ ([out, M] from weight [out, in] and tokens h2d [M, in]:
    the block's `in_proj.weight @ rearrange(h, "b l d -> d (b l)")`) with
    this module's products."""
    return _ProjTokensLastFn.apply(weight, h2d)
