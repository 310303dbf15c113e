"""Autograd functions of the Field block's elementwise work, forward and backward in one kernel each
(``csrc/train.hip``; canon:300-325, 1169-1173, 1193-1195, 1219-1221).

A backward that must itself be differentiable (``create_graph``) runs the stock ops instead, from the
tensors as they came in (saved before any copy for alignment, so that they keep their graph). Autograd
materialises the gradients of unused outputs as zeros, so that no backward sees a missing one.
"""
from __future__ import annotations

import torch
import torch.nn.functional as F

from . import _native as nat


def _stock_grads(fn, inputs, grads):
    """Differentiable gradients of ``fn(*inputs)``; ``inputs`` keep their place in the graph. Taken with
    respect to aliases: one input may depend on another (an output of the function whose backward this
    is does on its inputs), and the derivative wanted here is the partial one."""
    with torch.enable_grad():
        inputs = [t.view_as(t) for t in inputs]
        outs = fn(*inputs)
        outs = outs if isinstance(outs, tuple) else (outs,)
        pairs = [(o, g) for o, g in zip(outs, grads) if o.requires_grad]
        wanted = [t for t in inputs if t.requires_grad]
        got = iter(torch.autograd.grad([o for o, _ in pairs], wanted, [g for _, g in pairs], create_graph=True,
                                       allow_unused=True) if wanted else ())
    return [next(got) if t.requires_grad else None for t in inputs]


def _aligned(t: torch.Tensor) -> torch.Tensor:
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _workspace(lib, dim: int, device) -> torch.Tensor:
    return torch.empty(int(lib.fl_train_workspace_bytes(dim)), device=device, dtype=torch.uint8)


def _norm_ops(x, w, eps, dtype):
    return (x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + eps) * w).to(dtype)


class Norm(torch.autograd.Function):
    """RMSNorm of fp32 rows, written in the type its product reads."""

    @staticmethod
    def forward(ctx, x, w, eps, dtype):
        lib, dim = nat.load(), x.shape[-1]
        rows = x.numel() // dim
        rstd = torch.empty(rows, device=x.device, dtype=torch.float32)
        ctx.save_for_backward(x, w, rstd)
        x = _aligned(x)
        out = torch.empty(x.shape, device=x.device, dtype=dtype)
        nat.check(lib.fl_train_norm(nat.ptr(x), rows, dim, nat.ptr(w), eps, nat.ptr(out), nat.dtype_code(dtype),
                                    nat.ptr(rstd), nat.stream_handle(x.device)), "fl_train_norm")
        ctx.eps, ctx.dtype = eps, dtype
        return out

    @staticmethod
    def backward(ctx, gy):
        x, w, rstd = ctx.saved_tensors
        if torch.is_grad_enabled():
            return (*_stock_grads(lambda a, b: _norm_ops(a, b, ctx.eps, ctx.dtype), (x, w), (gy,)), None, None)
        lib, dim = nat.load(), x.shape[-1]
        x, gy = _aligned(x), _aligned(gy)
        gx, gw, ws = torch.empty_like(x), torch.empty_like(w), _workspace(lib, dim, x.device)
        nat.check(lib.fl_train_norm_backward(
            nat.ptr(gy), nat.dtype_code(gy.dtype), nat.ptr(x), rstd.numel(), dim, nat.ptr(w), nat.ptr(rstd),
            nat.ptr(gx), nat.ptr(gw), nat.ptr(ws), ws.numel(), nat.stream_handle(x.device)), "fl_train_norm_backward")
        return gx, gw, None, None


def _gate_norm_ops(x, out, gate, w, eps, dtype):
    x = x + (out * torch.sigmoid(gate)).to(x.dtype)
    return x, _norm_ops(x, w, eps, dtype)


class GateNorm(torch.autograd.Function):
    """(x + out * sigmoid(gate), its RMSNorm): fp32 residual, out and gate of one product type."""

    @staticmethod
    def forward(ctx, x, out, gate, w, eps, dtype):
        lib, dim, kept = nat.load(), x.shape[-1], (out, gate)
        x, out, gate = _aligned(x), _aligned(out), _aligned(gate)
        rows = x.numel() // dim
        x_new, normed = torch.empty_like(x), torch.empty(x.shape, device=x.device, dtype=dtype)
        rstd = torch.empty(rows, device=x.device, dtype=torch.float32)
        nat.check(lib.fl_train_gate_norm(
            nat.ptr(x), nat.ptr(out), nat.ptr(gate), nat.dtype_code(out.dtype), rows, dim, nat.ptr(w), eps,
            nat.ptr(x_new), nat.ptr(normed), nat.dtype_code(dtype), nat.ptr(rstd), nat.stream_handle(x.device)),
            "fl_train_gate_norm")
        # x itself is needed only by a differentiable backward: x_new = x + ... gives it back
        ctx.save_for_backward(x_new, *kept, w, rstd)
        ctx.eps, ctx.dtype = eps, dtype
        return x_new, normed

    @staticmethod
    def backward(ctx, g_x, g_normed):
        x_new, out, gate, w, rstd = ctx.saved_tensors
        if torch.is_grad_enabled():
            # through the norm from x_new, then through the gated sum, whose value x_new already is
            gx, gw = _stock_grads(lambda a, b: _norm_ops(a, b, ctx.eps, ctx.dtype), (x_new, w), (g_normed,))
            gx = g_x if gx is None else g_x + gx
            g_out, g_gate = _stock_grads(lambda o, g: (o * torch.sigmoid(g)).to(x_new.dtype), (out, gate), (gx,))
            return gx, g_out, g_gate, gw, None, None
        lib, dim = nat.load(), x_new.shape[-1]
        out, gate = _aligned(out), _aligned(gate)
        g_x, g_normed = _aligned(g_x), _aligned(g_normed)
        gx, g_out, g_gate, gw = (torch.empty_like(t) for t in (x_new, out, gate, w))
        ws = _workspace(lib, dim, x_new.device)
        nat.check(lib.fl_train_gate_norm_backward(
            nat.ptr(g_x), nat.ptr(g_normed), nat.dtype_code(g_normed.dtype), nat.ptr(x_new), nat.ptr(out),
            nat.ptr(gate), nat.dtype_code(out.dtype), rstd.numel(), dim, nat.ptr(w), nat.ptr(rstd), nat.ptr(gx),
            nat.ptr(g_out), nat.ptr(g_gate), nat.ptr(gw), nat.ptr(ws), ws.numel(),
            nat.stream_handle(x_new.device)), "fl_train_gate_norm_backward")
        return gx, g_out, g_gate, gw, None, None


def _swiglu_ops(gu):
    gate, up = gu.chunk(2, dim=-1)
    return F.silu(gate) * up


class Swiglu(torch.autograd.Function):
    """silu(gate) * up of the packed product [..., 2H]."""

    @staticmethod
    def forward(ctx, gu):
        lib = nat.load()
        ctx.save_for_backward(gu)
        gu = _aligned(gu)
        hidden = gu.shape[-1] // 2
        out = torch.empty((*gu.shape[:-1], hidden), device=gu.device, dtype=gu.dtype)
        nat.check(lib.fl_swiglu(nat.ptr(gu), nat.dtype_code(gu.dtype), gu.numel() // (2 * hidden), hidden,
                                nat.ptr(out), nat.stream_handle(gu.device)), "fl_swiglu")
        return out

    @staticmethod
    def backward(ctx, gy):
        gu, = ctx.saved_tensors
        if torch.is_grad_enabled():
            return _stock_grads(_swiglu_ops, (gu,), (gy,))[0]
        lib, hidden = nat.load(), gu.shape[-1] // 2
        gu, gy = _aligned(gu), _aligned(gy)
        out = torch.empty_like(gu)
        nat.check(lib.fl_swiglu_backward(nat.ptr(gu), nat.ptr(gy), nat.dtype_code(gu.dtype),
                                         gu.numel() // (2 * hidden), hidden, nat.ptr(out),
                                         nat.stream_handle(gu.device)), "fl_swiglu_backward")
        return out


def transition_ops(radius_logit, theta):
    """(tr, ti, gamma) of canon:1169-1173 in stock ops."""
    radius = torch.sigmoid(radius_logit).clamp(0.50, 0.99995).float()
    theta = theta.float()
    gamma = torch.sqrt((1.0 - radius.square()).clamp_min(1e-4))
    return (radius * torch.cos(theta)).contiguous(), (radius * torch.sin(theta)).contiguous(), gamma.contiguous()


class Transition(torch.autograd.Function):
    """The transition parameters, fp32 [C] each, from fp32 radius_logit and theta."""

    @staticmethod
    def forward(ctx, radius_logit, theta):
        lib, c = nat.load(), radius_logit.numel()
        out = [torch.empty_like(radius_logit) for _ in range(3)]
        nat.check(lib.fl_field_params(nat.ptr(radius_logit), nat.ptr(theta), c, None, 0, *[nat.ptr(t) for t in out],
                                      None, nat.stream_handle(theta.device)), "fl_field_params")
        ctx.save_for_backward(radius_logit, theta)
        return tuple(out)

    @staticmethod
    def backward(ctx, *grads):
        radius_logit, theta = ctx.saved_tensors
        if torch.is_grad_enabled():
            return tuple(_stock_grads(transition_ops, (radius_logit, theta), grads))
        lib, c = nat.load(), radius_logit.numel()
        grads = [g.contiguous() for g in grads]
        gl, gt = torch.empty_like(radius_logit), torch.empty_like(theta)
        nat.check(lib.fl_field_params_backward(nat.ptr(radius_logit), nat.ptr(theta), c, *[nat.ptr(g) for g in grads],
                                               nat.ptr(gl), nat.ptr(gt), nat.stream_handle(theta.device)),
                  "fl_field_params_backward")
        return gl, gt
