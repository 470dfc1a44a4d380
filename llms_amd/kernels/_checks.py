"""Argument checks shared by the fused-projection wrappers."""

from __future__ import annotations

import torch
from torch._C import _functorch
from torch.autograd import forward_ad
from torch.nn.modules import module as _module

from ._eager import RMSNorm


def require_bf16_hip(fn: str, **tensors: torch.Tensor) -> None:
    """The HIP kernels take bfloat16 activations/weights on a HIP device.

    Raises ``TypeError`` for another dtype and ``ValueError`` for a tensor that
    is not on a HIP device (there is no CPU or fp32 path).
    """
    for name, t in tensors.items():
        if t.dtype != torch.bfloat16:
            raise TypeError(f"{fn}: {name} must be torch.bfloat16, got {t.dtype}")
        if t.device.type != "cuda":
            raise ValueError(
                f"{fn}: {name} is on {t.device}; the fused projections run only on a "
                "HIP (ROCm) device"
            )


def require_device(fn: str, t: torch.Tensor, name: str) -> None:
    if t.device.type != "cuda":
        raise ValueError(
            f"{fn}: {name} is on {t.device}; the fused projections run only on a "
            "HIP (ROCm) device"
        )


def inner_contiguous(t: torch.Tensor) -> torch.Tensor:
    """t with unit stride along the last dim (the C ABI takes row strides)."""
    if t.dim() >= 1 and t.shape[-1] > 1 and t.stride(-1) != 1:
        return t.contiguous()
    return t


def plain_norm(m) -> bool:
    """Whether m is the RMSNorm of ``_eager.py`` with nothing attached to its
    call and no ``forward`` of its own set on it (a fused kernel may then
    normalise with its weight and eps)."""
    return (type(m) is RMSNorm and "forward" not in m.__dict__ and not m._forward_hooks and not m._forward_pre_hooks
            and not _module._global_forward_hooks and not _module._global_forward_pre_hooks)


def transformed(*tensors: torch.Tensor) -> bool:
    """Whether autograd, in either mode, or a torch.func transform (vmap, grad,
    jvp) may follow an operation on these. What torch does not say about its
    forward mode counts as yes."""
    return ((torch.is_grad_enabled() and any(t.requires_grad for t in tensors))
            or getattr(forward_ad, "_current_level", 0) >= 0
            or _functorch.peek_interpreter_stack() is not None)


def autocast() -> bool:
    """Whether torch's autocast would choose the types of a matmul here."""
    return torch.is_autocast_enabled("cuda")
