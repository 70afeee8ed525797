"""Autograd Functions over the fused residual-add + RMSNorm kernels
(mg_add_rmsnorm_fwd / mg_add_rmsnorm_bwd).

Reference semantics: torch.nn.RMSNorm(dim) as used by mingru/minLM.py:67,
:69, :74 (eps=None -> float32 machine epsilon) and the residual adds at
mingru/minLM.py:125 and :130. The residual stream is kept in fp32; the
normalized output is produced in the activation dtype, optionally (bf16) as
a hi/lo pair [N, 2D] = [bf16(y) | bf16(y - bf16(y))] whose hi half is the
usual output: the operand of the fp32-accurate products (gemm HILO).
Weights of any floating dtype are accepted (a model cast with
.to(torch.bfloat16), as reference generate.py:140-142 does); the kernels read
them as fp32.
"""
import torch

from ._lib import MG_BF16, dtype_code, native, require_cuda, stream_of

FP32_EPS = float(torch.finfo(torch.float32).eps)


def _fwd(x, delta, w, out_dtype, with_lo=False):
    """Returns (x_out, y, rstd, pair): pair is the [..., 2D] hi/lo buffer
    (y is its first half) when with_lo, else None."""
    require_cuda(x, delta, w)
    return native().norm_fwd(x, delta, w, dtype_code(out_dtype) == MG_BF16, with_lo, stream_of(x))


def _bwd(xn, w, rstd, dy, dres, want_dx, delta_dtype, want_ddelta):
    return native().norm_bwd(xn, w, rstd, dy, dres, want_dx, dtype_code(delta_dtype) if want_ddelta else -1, None,
                             stream_of(xn))


class RMSNormResidualFn(torch.autograd.Function):
    """(x, rmsnorm(x) * w) for an fp32 x that also continues as the residual
    stream: the gradient reaching x through the residual joins the norm's
    gradient inside the backward kernel instead of in a separate add."""

    @staticmethod
    def forward(ctx, x, w, out_dtype, with_lo):
        _, y, rstd, pair = _fwd(x, None, w, out_dtype, with_lo)
        ctx.save_for_backward(x, w, rstd)
        ctx.set_materialize_grads(False)
        if pair is not None:
            ctx.mark_non_differentiable(pair)
        return x.view_as(x), y, pair

    @staticmethod
    def backward(ctx, dx_res, dy, _dpair):
        x, w, rstd = ctx.saved_tensors
        if dx_res is None and dy is None:
            return None, None, None, None
        dx, _, dw = _bwd(x, w, rstd, dy, dx_res, ctx.needs_input_grad[0], None, False)
        return dx, (dw if ctx.needs_input_grad[1] else None), None, None


class RMSNormFn(torch.autograd.Function):
    """y = x * w / sqrt(mean(x^2) + eps) over the last dim; x fp32, y in out_dtype."""

    @staticmethod
    def forward(ctx, x, w, out_dtype):
        _, y, rstd, _ = _fwd(x, None, w, out_dtype)
        ctx.save_for_backward(x, w, rstd)
        return y

    @staticmethod
    def backward(ctx, dy):
        x, w, rstd = ctx.saved_tensors
        dx, _, dw = _bwd(x, w, rstd, dy, None, ctx.needs_input_grad[0], None, False)
        return dx, (dw if ctx.needs_input_grad[1] else None), None


class AddRMSNormFn(torch.autograd.Function):
    """(x + delta, rmsnorm(x + delta) * w): the residual add fused with the next norm."""

    @staticmethod
    def forward(ctx, x, delta, w, out_dtype, with_lo):
        x_out, y, rstd, pair = _fwd(x, delta, w, out_dtype, with_lo)
        ctx.save_for_backward(x_out, w, rstd)
        ctx.delta_dtype = delta.dtype
        ctx.set_materialize_grads(False)  # an unused x_out (the final norm's) gets no zero tensor
        if pair is not None:
            ctx.mark_non_differentiable(pair)
        return x_out, y, pair

    @staticmethod
    def backward(ctx, dx_out, dy, _dpair):
        xn, w, rstd = ctx.saved_tensors
        if dx_out is None and dy is None:
            return None, None, None, None, None
        want_dx, want_dd = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        dx, dd, dw = _bwd(xn, w, rstd, dy, dx_out, want_dx, ctx.delta_dtype, want_dd)
        return dx, dd, (dw if ctx.needs_input_grad[2] else None), None, None


def _check(x, w, delta=None):
    """Validates the operands; returns the weight as fp32 (a cast that autograd
    differentiates, for models whose parameters are bf16 or fp16)."""
    require_cuda(x, w, delta)
    if x.dtype != torch.float32:
        raise ValueError(f"the residual stream must be float32, got {x.dtype}")
    if not w.is_floating_point() or w.dim() != 1 or w.shape[0] != x.shape[-1]:
        raise ValueError(f"weight must be a floating [{x.shape[-1]}] vector, got {w.dtype} {tuple(w.shape)}")
    if delta is not None and delta.shape != x.shape:
        raise ValueError(f"delta {tuple(delta.shape)} must match x {tuple(x.shape)}")
    return w if w.dtype == torch.float32 else w.float()


def _lo_ok(out_dtype, with_lo):
    if with_lo and out_dtype != torch.bfloat16:
        raise ValueError("the hi/lo pair output needs a bfloat16 output")
    return with_lo


def rms_norm(x, w, out_dtype=None):
    """RMSNorm of an fp32 tensor over its last dim with fp32 epsilon; output in out_dtype."""
    w = _check(x, w)
    return RMSNormFn.apply(x.contiguous(), w, out_dtype or x.dtype)


def rms_norm_residual(x, w, out_dtype=None, with_lo=False):
    """Returns (x, rms_norm(x, w), pair) where the first output carries x on as
    the residual stream (one backward kernel for both uses of x); pair is the
    hi/lo buffer when with_lo (bf16 output; the second output is its hi half),
    else None."""
    w = _check(x, w)
    out_dtype = out_dtype or x.dtype
    return RMSNormResidualFn.apply(x.contiguous(), w, out_dtype, _lo_ok(out_dtype, with_lo))


def add_rms_norm(x, delta, w, out_dtype=None, with_lo=False):
    """Returns (x + delta, rms_norm(x + delta, w), pair); x fp32, delta fp32 or
    bf16; pair as in rms_norm_residual."""
    w = _check(x, w, delta)
    out_dtype = out_dtype or x.dtype
    return AddRMSNormFn.apply(x.contiguous(), delta.contiguous(), w, out_dtype, _lo_ok(out_dtype, with_lo))
