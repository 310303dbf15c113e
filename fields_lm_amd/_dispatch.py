"""When a block may run its hand-written kernels in place of the stock ops.

The kernels are called through raw pointers, outside PyTorch's dispatcher, so whatever observes or
transforms operators there (autograd, tracing, vmap, forward-mode derivatives, dispatch modes, tensor
subclasses) keeps the stock ops.
"""
from __future__ import annotations

import torch
import torch.nn as nn
from torch.autograd import forward_ad

KERNEL_DTYPES = (torch.bfloat16, torch.float32)


def eager(*tensors: torch.Tensor) -> bool:
    """Plain device tensors on one device, and nothing that watches or transforms their operators."""
    if (torch.compiler.is_compiling() or torch.jit.is_tracing() or forward_ad._current_level >= 0
            or torch._C._len_torch_dispatch_stack() > 0):
        return False
    device = tensors[0].device
    return device.type == "cuda" and all(
        type(t) in (torch.Tensor, nn.Parameter) and t.device == device
        and not torch._C._functorch.is_functorch_wrapped_tensor(t) for t in tensors)


def no_grad_needed(*tensors: torch.Tensor) -> bool:
    return not torch.is_grad_enabled() or not any(t.requires_grad for t in tensors)


def plain_call(module: nn.Module, cls: type) -> bool:
    """``module`` is exactly ``cls`` and calling it is nothing but its forward: no hook, no replaced
    forward."""
    m, own = nn.modules.module, module.__dict__
    return (type(module) is cls and "forward" not in own
            and not (own["_forward_hooks"] or own["_forward_pre_hooks"] or own["_backward_hooks"]
                     or own["_backward_pre_hooks"] or m._global_forward_hooks or m._global_forward_pre_hooks))


def plain_linear(layer: nn.Module) -> bool:
    """An nn.Linear whose call is nothing but its GEMM on an ordinary weight."""
    if not plain_call(layer, nn.Linear):
        return False
    weight = layer._parameters.get("weight")  # (an attribute of the module costs ten times a dict's entry)
    return type(layer.weight if weight is None else weight) in (nn.Parameter, torch.Tensor)


def free_rounding() -> bool:
    """Whether kernels may run that round or sum in another order than the stock ops they replace.

    Not under autocast. There the types of a block's products are autocast's to choose, and it is
    how the whole model runs: 24 bf16 layers grow one changed rounding to 2e-2 of the logits, which
    turns near ties of a greedy continuation into other tokens (measured with the Mamba-2 kernels:
    several of 64 streams differed after one token). So a generation loop under autocast keeps
    every bit; kernels that give the stock bits run there too. ``cast_for_inference`` weights need
    no autocast, and without it every kernel runs."""
    return not torch.is_autocast_enabled()
