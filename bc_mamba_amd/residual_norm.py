"""The leaky residual and its layer norm between two blocks
(lra_impl.py:1381-1427): v' = alpha v + dv, h = norm(v').

On the GPU in fp32 both run as one kernel each way (bcm_residual_norm_fwd /
_bwd); everything else is torch's."""
import torch

try:
    from . import _native as _nat
except ImportError:  # imported with this directory on sys.path
    import _native as _nat

__all__ = ["layer_norm", "residual_norm"]

_PLAIN = (torch.Tensor, torch.nn.Parameter)
MAX_DIM = 1024


def _plain_module(m, cls):
    """m is a cls whose call is exactly its class's forward: no hooks of its
    own, no replaced forward."""
    return (type(m) is cls and "forward" not in vars(m) and not m._forward_hooks and not m._forward_pre_hooks
            and not m._backward_hooks and not m._backward_pre_hooks)


def _plain_mode():
    """Nothing that must see the single operations: tracing, autocast, vmap
    and the other function transforms, forward-mode gradients, hooks on every
    module."""
    g = torch.nn.modules.module
    return not (torch.compiler.is_compiling() or torch.is_autocast_enabled("cuda")
                or torch._C._functorch.peek_interpreter_stack() is not None
                or torch.autograd.forward_ad._current_level >= 0
                or g._global_forward_hooks or g._global_forward_pre_hooks
                or g._global_backward_hooks or g._global_backward_pre_hooks)


def _kernel_ok(norm, x, *more):
    """The kernels apply to norm (a LayerNorm over x's last dimension with
    weight and bias) and the contiguous fp32 tensors x and more."""
    if not _plain_module(norm, torch.nn.LayerNorm) or not _plain_mode():
        return False
    w, b, D = norm.weight, norm.bias, norm.normalized_shape[-1]
    if w is None or b is None or len(norm.normalized_shape) != 1 or D % 4 or not 4 <= D <= MAX_DIM:
        return False
    if x.dim() < 1 or x.size(-1) != D or x.numel() == 0 or x.numel() >= 2 ** 31:
        return False
    return all(type(t) in _PLAIN and t.dtype == torch.float32 and t.is_cuda and t.device == x.device
               and t.is_contiguous() and t.data_ptr() % 16 == 0 for t in (x, w, b, *more)) \
        and all(t.shape == x.shape for t in more)


def _dense(g):
    """g contiguous and aligned for the kernel's 16-byte loads (or None)."""
    if g is None or (g.is_contiguous() and g.data_ptr() % 16 == 0):
        return g
    return g.clone(memory_format=torch.contiguous_format)


class _ResidualNormFn(torch.autograd.Function):
    """(h, v') of v (or None: the norm of dv alone, v' = dv) and dv."""

    @staticmethod
    def forward(ctx, v, dv, weight, bias, alpha: float, eps: float):
        D, rows = dv.size(-1), dv.numel() // dv.size(-1)
        h = torch.empty_like(dv)
        v_out = torch.empty_like(dv) if v is not None else None
        mean, rstd = (torch.empty(rows, dtype=dv.dtype, device=dv.device) for _ in range(2))
        with _nat.on_device(dv.device):
            _nat.call("bcm_residual_norm_fwd", _nat.ptr(v), dv.data_ptr(), alpha, weight.data_ptr(), bias.data_ptr(),
                      rows, D, eps, _nat.ptr(v_out), h.data_ptr(), mean.data_ptr(), rstd.data_ptr(),
                      _nat.stream_of(dv))
        ctx.alpha, ctx.eps, ctx.residual = alpha, eps, v is not None
        ctx.save_for_backward(v_out if v is not None else dv, weight, mean, rstd)
        ctx.set_materialize_grads(False)
        return h, v_out

    @staticmethod
    def backward(ctx, gh, gv):
        x, weight, mean, rstd = ctx.saved_tensors
        alpha, residual = ctx.alpha, ctx.residual
        # the residual alone, a graph of the gradients asked for, or a batch of gradients at once
        if gh is None or torch.is_grad_enabled() or _nat.no_memory(gh, gv):
            d, dw, db = gv, None, None
            if gh is not None:
                mu = x.mean(-1, keepdim=True)
                xc = x - mu
                rs = torch.rsqrt(xc.pow(2).mean(-1, keepdim=True) + ctx.eps)
                xh, g = xc * rs, gh * weight
                d = rs * (g - g.mean(-1, keepdim=True) - xh * (g * xh).mean(-1, keepdim=True))
                d = d if gv is None else d + gv
                dw, db = ((t.reshape(-1, t.size(-1))).sum(0) for t in (gh * xh, gh))
            return (d * alpha if residual and d is not None else None), d, dw, db, None, None
        gh, gv = _dense(gh), _dense(gv)
        D, rows = x.size(-1), mean.numel()
        d, dw, db = torch.empty_like(x), torch.empty_like(weight), torch.empty_like(weight)
        dv = torch.empty_like(x) if residual and ctx.needs_input_grad[0] else None
        with _nat.on_device(x.device):
            nbytes = int(_nat.lib().bcm_residual_norm_workspace_bytes(rows, D))
            ws = torch.empty(nbytes // 4, dtype=torch.float32, device=x.device)
            _nat.call("bcm_residual_norm_bwd", gh.data_ptr(), _nat.ptr(gv), x.data_ptr(), alpha, weight.data_ptr(),
                      mean.data_ptr(), rstd.data_ptr(), rows, D, d.data_ptr(), _nat.ptr(dv), dw.data_ptr(),
                      db.data_ptr(), ws.data_ptr(), nbytes, _nat.stream_of(x))
        return dv, d, dw, db, None, None


def residual_norm(norm, v, dv, alpha):
    """(norm(v'), v') with v' = alpha * v + dv."""
    if type(alpha) is float and _kernel_ok(norm, v, dv):
        return _ResidualNormFn.apply(v, dv, norm.weight, norm.bias, alpha, float(norm.eps))
    v_out = alpha * v + dv
    return norm(v_out), v_out


def layer_norm(norm, x):
    """norm(x)."""
    if _kernel_ok(norm, x):
        return _ResidualNormFn.apply(None, x, norm.weight, norm.bias, 1.0, float(norm.eps))[0]
    return norm(x)
