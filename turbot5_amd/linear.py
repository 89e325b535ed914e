"""Linear layers of a training step with fp32 weights, on the bf16 matrix cores (``t5a_gemm_f32``).

The reference runs its linear layers in torch (src/turbot5/model/attentions.py:59-62, modules.py); in fp32 those are
products on the fp32 matrix cores, four fifths of a training step's time.  ``t5a_gemm_f32`` forms the same products from
operands split into three bf16 parts, as accurately and in less time, several of one shape in one launch, and rounds its
result to the attention's type, applies ReLU or its derivative on the way out.
"""
from __future__ import annotations

import torch
from torch import nn

from .ops import _nodes, _plain

MAX_BYTES = 0x7fe00000      # of an operand, which the kernel reads with 32-bit offsets


def _gemm(a, b, out, a_trans=False, b_trans=False, sum_groups=False, alpha=1.0, relu=False, positive=None):
    """out[g] = alpha_g a[g] b[g]^T over lists of two-dimensional contiguous tensors (see include/t5attn.h): the call that the nodes of
    ``project`` and ``feed_forward_relu`` make."""
    _nodes().gemm(a, b, out, bool(a_trans), bool(b_trans), bool(sum_groups), bool(relu), float(alpha), positive)
    return out


def _full_precision() -> bool:
    """torch's own fp32 products would be fp32 ones: neither autocast nor a faster precision has been asked for."""
    if torch.is_autocast_enabled("cuda"):
        return False
    try:
        return torch.get_float32_matmul_precision() == "highest" and not torch.backends.cuda.matmul.allow_tf32
    except RuntimeError:      # (set through torch's older and newer switches at once)
        return False


def _bare(m: nn.Module) -> bool:
    """A linear layer that is its weight and nothing else: no subclass, hook, patch or bias."""
    return (type(m) is nn.Linear and m.bias is None and "forward" not in m.__dict__
            and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks))


def takes(x: torch.Tensor, *layers: nn.Module) -> bool:
    """Whether these layers' products over ``x`` (fp32, or bf16 that torch would widen) are part of a training step that
    ``project`` takes: fp32 weights of one shape on x's device and plain reverse-mode autograd.  Any number of rows: at 8 a product of a T5-small
    layer takes 4 to 12 us, the library's fp32 one 19 to 25; at 4500 all of a layer's take 600 us, the library's 900."""
    if not x.is_cuda or not torch.is_grad_enabled() or not all(_bare(m) for m in layers):
        return False
    weights = [m.weight for m in layers]
    first = weights[0]
    return (_plain(x, *weights) and (x.requires_grad or any(w.requires_grad for w in weights))
            and x.dtype in (torch.float32, torch.bfloat16) and x.dim() >= 2
            and x.numel() > 0 and x.shape[-1] == first.shape[1]
            and all(w.dtype == torch.float32 and w.device == x.device and w.shape == first.shape for w in weights)
            and first.shape[0] % 8 == 0 and first.shape[1] % 8 == 0 and first.numel() > 0
            and x.numel() * 4 < MAX_BYTES and x.numel() // x.shape[-1] * first.shape[0] * 4 < MAX_BYTES
            and first.numel() * 4 < MAX_BYTES
            and _full_precision() and not nn.modules.module._has_any_global_hook()
            and all(type(m) is torch.utils._device.DeviceContext for m in torch.overrides._get_current_function_mode_stack()))


def widths_chain(wi: nn.Module, wo: nn.Module) -> bool:
    """wo is a layer of the same kind over wi's output (which ``takes`` has said yes to), no wider than wi's input: then its weight and its
    results are no larger than what ``takes`` has measured."""
    return (_bare(wo) and _plain(wo.weight) and wo.weight.dtype == torch.float32 and wo.weight.device == wi.weight.device
            and wo.weight.shape[1] == wi.weight.shape[0] and wo.weight.shape[0] % 8 == 0 and 0 < wo.weight.shape[0] <= wi.weight.shape[1])


def project(x, dtype, factor, *layers):
    """x W_0^T * factor, x W_1^T, ...: products of the same rows with up to three weights of one shape, each result rounded to
    ``dtype`` once, in x's shape; ``takes`` has said yes."""
    out = _nodes().project(x.reshape(-1, x.shape[-1]), dtype, float(factor), [m.weight for m in layers])
    return [t.view(*x.shape[:-1], t.shape[-1]) for t in out]


def feed_forward_relu(x, wi: nn.Linear, wo: nn.Linear):
    """relu(wi(x)) through wo, ReLU and its derivative part of the products that make their operand; ``takes`` and
    ``widths_chain`` have said yes."""
    return _nodes().feed_forward_relu(x.reshape(-1, x.shape[-1]), wi.weight, wo.weight).view(*x.shape[:-1], wo.weight.shape[0])
