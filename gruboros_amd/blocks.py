"""Block-level autograd functions of the bf16 minLM training path.

Reference mingru/minLM.py:107-149: per layer
    x = minGRU(RMSNorm(x)) + x        (:119-125)
    x = FeedForward(RMSNorm(x)) + x   (:127-130)
then the final RMSNorm, the logits and the cross-entropy (:137-149).

Here each of those three pieces is one torch.autograd.Function (bf16
activations over fp32 master weights):

  MinGRUBlock   x1 = x + pending; n = RMSNorm(x1) as a hi/lo pair;
                hg = [n W_h^T (fp32-accurate) | n W_g^T]; h = scan(hg) in fp32;
                expansion 1: the scan writes x2 = x1 + h itself (h is kept only as
                fp32 checkpoints); else out = to_out(h) (fp32-accurate).
  FFBlock       x2 = x1 + out (or x2 as given); n2 = RMSNorm(x2);
                pending = FeedForward(n2) (bf16).
  FinalNormCE   embed = RMSNorm(x + pending); mean cross-entropy of
                embed W_out^T (streaming loss kernel).

Why blocks rather than one Function per op: every gradient a block stores
in bf16 (dlogits, the input-gradient products, dgate/dhidden, dpre, the
FeedForward output's gradient) is rounded stochastically by the kernel that
writes it. An autograd boundary at a bf16 tensor would instead cast its
incoming gradient to bf16 with round-to-nearest, whose errors at a near-
uniform softmax repeat across the rows of a label and add up in the weight
gradients (measured on the fp64 restatement: 4-7% at the cfg3 row count
against 0.5% with stochastic rounding). The gradients crossing block boundaries
are the fp32 residual stream's, the fp32 minGRU output's, and the bf16
FeedForward output's (stochastically rounded by the next block's norm).

The launches of a block pass are issued by one call into csrc/host/native.cpp.
"""
import torch

from . import _lib
from .linear import bf16_copy, bf16_pair, grad_target
from .scan import _workspace as _scan_workspace

BF16 = torch.bfloat16

# The FeedForward's two weight gradients in one K-split launch
# (mg_gemm_wgrad_pair) instead of one launch each; likewise to_out's and
# to_hidden_and_gate's (expansion != 1).
FF_DW_PAIR = True

# At expansion 1 the scan adds its state to the residual stream itself
# (mg_scan_fwd_residual) and keeps h only as fp32 checkpoints for the backward;
# False: the scan writes h and the FeedForward's norm adds it.
SCAN_RESIDUAL = True

# to_hidden_and_gate's forward as one launch (mg_gemm_hilo_prefix: the hidden
# half's tiles hi/lo, the gate half's plain) instead of two.
HG_ONE_LAUNCH = True


def _f32(b):
    """A bias as the fp32 contiguous vector the GEMM epilogue adds."""
    return b if b.dtype == torch.float32 and b.is_contiguous() else b.float().contiguous()


class MinGRUBlock(torch.autograd.Function):
    """(x, pending) -> (x_next, out, h_last); see the module docstring.

    x: fp32 [B, T, D] residual stream; pending: bf16 [B, T, D] (the previous
    FeedForward's output, not yet added) or None; w_norm fp32 [D]; w_hg fp32
    master [2 Di, D]; h0 fp32 [B, Di] or None; w_to fp32 master [D, Di] or None.
    Without to_out (expansion 1): x_next = x + pending + h (the scan adds its
    state to the residual stream) and out is None. With it: x_next = x + pending
    and out = to_out(h), fp32 [B, T, D]. h_last fp32 [B, 1, Di]."""

    @staticmethod
    def forward(ctx, x, pending, w_norm, w_hg, h0, w_to):
        ctx.set_materialize_grads(False)
        B, T, D = x.shape
        N, Di = B * T, w_hg.shape[0] // 2
        ctx.w_hg, ctx.w_to = w_hg, w_to  # for their .grad (weight gradients added in place, grad_target)
        _lib.require_cuda(x, pending, w_norm, w_hg, h0, w_to)
        x2 = x.reshape(N, D)
        whp = bf16_pair(w_hg)
        whb = bf16_copy(w_hg)
        x_out, rstd, pair, hg, h, h_last, out, h_pair, ckpt = _lib.native().gru_forward(
            x2, pending.reshape(N, D) if pending is not None else None, w_norm, whp, whb,
            bf16_pair(w_to) if w_to is not None else None, h0, B, T, SCAN_RESIDUAL, HG_ONE_LAUNCH,
            _scan_workspace(x.device, B, T, Di), _lib.stream_of(x))
        xn = x_out if x_out is not None else x2
        ctx.save_for_backward(xn, w_norm, rstd, pair, hg, h, h0, whb, ckpt, h_pair,
                              bf16_copy(w_to) if w_to is not None else None)
        ctx.dims = (B, T, D, Di)
        ctx.has_pending = pending is not None
        if w_to is None and ckpt is not None:  # expansion 1: x_next = x1 + h, h kept as checkpoints
            return out, None, h_last
        x1 = x_out.view(B, T, D) if x_out is not None else x.view_as(x)
        return x1, out, h_last

    @staticmethod
    def backward(ctx, dx1, dout, dh_last):
        B, T, D, Di = ctx.dims
        xn, w_norm, rstd, pair, hg, h, h0, whb, ckpt, h_pair, wtb = ctx.saved_tensors
        want_hg, want_to = ctx.needs_input_grad[3], ctx.needs_input_grad[5]
        dx, dpend, dw_norm, dW_hg, dh0, dW_to = _lib.native().gru_backward(
            xn, w_norm, rstd, pair, hg, h, h0, whb, ckpt, h_pair, wtb, dx1, dout, dh_last, B, T, ctx.has_pending, want_hg,
            want_to, h0 is not None and ctx.needs_input_grad[4], FF_DW_PAIR, grad_target(ctx.w_hg) if want_hg else None,
            grad_target(ctx.w_to) if want_to else None, _scan_workspace(xn.device, B, T, Di), _lib.stream_of(xn))
        return (dx.view(B, T, D), dpend.view(B, T, D) if dpend is not None else None,
                dw_norm if ctx.needs_input_grad[2] else None, dW_hg,
                dh0.reshape(h0.shape) if dh0 is not None else None, dW_to)


class FFBlock(torch.autograd.Function):
    """(x1, out) -> (x2 = x1 + out, pending = FeedForward(RMSNorm(x2))).

    x1 fp32 [B, T, D]; out fp32 [B, T, D] (the minGRU branch), or None when
    x1 already holds it (then x2 is x1, returned as is); FeedForward =
    Linear(D, F) -> GELU -> Linear(F, D) (reference mingru/minLM.py:17-23)
    with fp32 masters; pending bf16. Forward and backward products run on
    mg_gemm: the first with the bias + GELU epilogue (pre-activation and
    activation written in one pass), the second with the bias epilogue."""

    @staticmethod
    def forward(ctx, x1, out, w_norm, w1, b1, w2, b2):
        ctx.set_materialize_grads(False)
        B, T, D = x1.shape
        N = B * T
        ctx.w1, ctx.w2 = w1, w2  # for their .grad (weight gradients added in place, grad_target)
        _lib.require_cuda(x1, out, w_norm, w1, b1, w2, b2)
        x1r = x1.reshape(N, D)
        w1b, w2b = bf16_copy(w1), bf16_copy(w2)
        x2, n2, rstd, pre, act, pend = _lib.native().ff_forward(
            x1r, out.reshape(N, D) if out is not None else None, w_norm, w1b, _f32(b1), w2b, _f32(b2), _lib.stream_of(x1))
        ctx.has_out = out is not None
        ctx.save_for_backward(x2 if x2 is not None else x1r, w_norm, rstd, n2, pre, act, w1b, w2b)
        ctx.dims = (B, T, D)
        return (x2.view(B, T, D) if ctx.has_out else x1), pend.view(B, T, D)

    @staticmethod
    def backward(ctx, dx2, dpend):
        B, T, D = ctx.dims
        N = B * T
        x2, w_norm, rstd, n2, pre, act, w1b, w2b = ctx.saved_tensors
        nat, stream = _lib.native(), _lib.stream_of(x2)
        dW1 = db1 = dW2 = db2 = None
        if dpend is None:
            dres = dx2.reshape(N, D) if dx2 is not None else None
            dx1, _, dw_norm = nat.norm_bwd(x2, w_norm, rstd, None, dres, True, -1, None, stream)
        else:
            dp = dpend.reshape(N, D)
            if dp.dtype != BF16 or not dp.is_contiguous():
                dp = dp.to(BF16).contiguous()
            dx1, dw_norm, dW1, db1, dW2, db2 = nat.ff_backward(x2, w_norm, rstd, n2, pre, act, w1b, w2b, dx2, dp, FF_DW_PAIR,
                                                               grad_target(ctx.w1), grad_target(ctx.w2), stream)
        # x2 = x1 + out: both inputs get the same gradient, written once and returned for both
        # (the consumer, MinGRUBlock.backward, only reads them)
        return dx1.view(B, T, D), (dx1.view(B, T, D) if ctx.has_out else None), dw_norm, dW1, db1, dW2, db2


class FinalNormCE(torch.autograd.Function):
    """mean CE(RMSNorm(x + pending) W_out^T, labels) (reference mingru/minLM.py:137-149)
    for V <= 256 classes on the streaming loss kernel (logits never in memory).
    x fp32 [B, T, D], pending bf16 [B, T, D] or None, labels int64 [B, T]."""

    @staticmethod
    def forward(ctx, x, pending, w_norm, w_out, labels):
        B, T, D = x.shape
        N = B * T
        _lib.require_cuda(x, pending, w_norm, w_out, labels)
        x2 = x.reshape(N, D)
        wob = bf16_copy(w_out)
        loss, x_out, embed, rstd, dl = _lib.native().head_forward(
            x2, pending.reshape(N, D) if pending is not None else None, w_norm, wob, labels.reshape(-1).contiguous(),
            _lib.stream_of(x))
        ctx.save_for_backward(x_out if x_out is not None else x2, w_norm, rstd, embed, dl, wob)
        ctx.dims = (B, T, D)
        ctx.has_pending = pending is not None
        return loss

    @staticmethod
    def backward(ctx, g):
        B, T, D = ctx.dims
        xn, w_norm, rstd, embed, dl, wob = ctx.saved_tensors
        # the logits gradient's product stays unscaled: the norm backward applies g as it loads it
        dx, dpend, dw_norm, dW = _lib.native().head_backward(xn, w_norm, rstd, embed, dl, wob, g, ctx.has_pending,
                                                             ctx.needs_input_grad[3], _lib.stream_of(xn))
        return (dx.view(B, T, D), dpend.view(B, T, D) if dpend is not None else None,
                dw_norm if ctx.needs_input_grad[2] else None, dW, None)


def supported(model):
    """Whether the block path applies: bf16 activations over fp32 masters, no
    conv, no dropout, a loss head the streaming kernel takes, and widths every
    product and kernel of the blocks takes (D, Di = D * expansion and the
    FeedForward's F multiples of 8; mg_gemm's N and K, the scan's Di % 4)."""
    D = model.dim
    V = model.to_logits.weight.shape[0]
    return (all(conv is None and dropout is None for conv, _, _, _, _, dropout in model.layers)
            and model.token_emb.weight.dtype == torch.float32 and D % 8 == 0 and V % 8 == 0 and V <= 256
            and all(gru.to_hidden_and_gate.weight.shape[0] % 16 == 0 and ff[0].weight.shape[0] % 8 == 0
                    for _, _, gru, _, ff, _ in model.layers))
