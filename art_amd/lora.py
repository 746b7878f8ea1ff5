"""LoRA linear layer on the MI355X kernels.

``LoRALinear`` is the counterpart of the peft ``lora.Linear`` module that the
reference installs on the attention and MLP projections
(src/art/local/state.py:86-92; defaults r = 8, alpha = 16, no dropout,
``bias="none"``: src/art/dev/model.py:52-67).  The base weight is frozen, and so
is the base layer's own bias when it has one (Qwen2.5's q/k/v projections do;
peft keeps it and ``bias="none"`` means it is not trained); only ``lora_A`` and
``lora_B`` receive gradients."""
from __future__ import annotations

import math

import torch
from torch import nn

from . import _lib, ops


def _frozen_bias(bias):
    if bias is None:
        return None
    if bias.requires_grad:
        raise ValueError("the bias of a LoRA-wrapped linear is frozen (peft bias='none'); got requires_grad=True")
    return bias.detach().to(torch.bfloat16).contiguous()


def _lora_projections(x, weights, lora_As, lora_Bs, scale: float, biases):
    """Projections of the same x through the native autograd function (art_amd/csrc/native_ops.cpp): one call
    each way, nothing concatenated.  The transposed copies of the frozen weights go along if there are any; the
    backward makes them on its first use otherwise."""
    graph = torch.is_grad_enabled() and any(t.requires_grad for t in (x, *lora_As, *lora_Bs))
    wts = [ops.known_transpose(w) for w in weights] if graph else []
    if any(wt is None for wt in wts):
        wts = []
    return _lib.native().lora_multi(x, weights, wts, lora_As, lora_Bs, biases, scale)


def lora_linear(x, weight, lora_A, lora_B, scale: float, bias=None):
    """y = x W^T + bias + scale * (x A^T) B^T with gradients for x, A and B (W and bias frozen)."""
    bias = _frozen_bias(bias)
    if not isinstance(weight, torch.Tensor):   # an NF4Weight: the bf16 weight lives inside each call only
        w = weight
        return _lib.native().lora_nf4(x, w.packed, w.absmax, w.absmax_q, w.code2, w.absmax2, float(w.offset),
                                      w.blocksize, *w.shape, lora_A, lora_B, bias, float(scale))
    return _lora_projections(x, [weight], [lora_A], [lora_B], float(scale), [bias])[0]


class LoRALinear(nn.Module):
    """Frozen bf16 linear with a trainable rank-r update; forward(x) -> y."""

    def __init__(self, in_features: int, out_features: int, r: int = 8, lora_alpha: int = 16,
                 device=None, dtype=torch.bfloat16, bias: bool = False):
        super().__init__()
        self.in_features, self.out_features, self.r = in_features, out_features, r
        self.scaling = lora_alpha / r
        self.weight = nn.Parameter(torch.empty(out_features, in_features, device=device, dtype=torch.bfloat16),
                                   requires_grad=False)
        self.bias = (nn.Parameter(torch.zeros(out_features, device=device, dtype=torch.bfloat16), requires_grad=False)
                     if bias else None)
        self.lora_A = nn.Parameter(torch.empty(r, in_features, device=device, dtype=dtype))
        self.lora_B = nn.Parameter(torch.zeros(out_features, r, device=device, dtype=dtype))
        self.reset_parameters()

    def reset_parameters(self) -> None:
        nn.init.normal_(self.weight, std=0.02)
        nn.init.kaiming_uniform_(self.lora_A, a=math.sqrt(5))  # peft's default for A; B starts at zero
        nn.init.zeros_(self.lora_B)

    @classmethod
    def from_linear(cls, linear: nn.Linear, r: int = 8, lora_alpha: int = 16) -> "LoRALinear":
        mod = cls(linear.in_features, linear.out_features, r, lora_alpha, device=linear.weight.device,
                  bias=linear.bias is not None)
        with torch.no_grad():
            mod.weight.copy_(linear.weight.to(torch.bfloat16))
            if linear.bias is not None:
                mod.bias.copy_(linear.bias.to(torch.bfloat16))
        return mod

    @classmethod
    def from_nf4(cls, w_nf4, r: int = 8, lora_alpha: int = 16, bias=None) -> "LoRALinear":
        """Wrap a frozen weight that stays in its 4-bit storage form (art_amd.quant.NF4Weight): the
        module then holds no 16-bit copy of it, as with `load_in_4bit=True` in the reference
        (src/art/dev/model.py:29)."""
        n_out, n_in = w_nf4.shape
        dev = w_nf4.packed.device
        mod = cls.__new__(cls)
        nn.Module.__init__(mod)
        mod.in_features, mod.out_features, mod.r = n_in, n_out, r
        mod.scaling = lora_alpha / r
        mod.weight = None
        mod.weight_nf4 = w_nf4
        mod.bias = (nn.Parameter(bias.detach().to(torch.bfloat16).to(dev), requires_grad=False)
                    if bias is not None else None)
        mod.lora_A = nn.Parameter(torch.empty(r, n_in, device=dev, dtype=torch.bfloat16))
        mod.lora_B = nn.Parameter(torch.zeros(n_out, r, device=dev, dtype=torch.bfloat16))
        nn.init.kaiming_uniform_(mod.lora_A, a=math.sqrt(5))
        return mod

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        weight = self.weight if self.weight is not None else self.weight_nf4
        return lora_linear(x, weight, self.lora_A, self.lora_B, self.scaling, self.bias)


class FusedLoRALinear(nn.Module):
    """Projections that read the same activations (q/k/v, or gate/up) in one call each way:
    one persistent launch over the tiles of all of them (the narrow projections, k and v with
    256 or 512 columns, ride along with the wide one instead of leaving most of the GPU idle),
    one accumulation for the input gradient, one pass over x for all dA.  ``forward(x)``
    returns the tuple of the individual outputs.  The module holds the given layers and
    nothing else: no second copy of the frozen weights, no stacked adapters."""

    def __init__(self, layers):
        super().__init__()
        layers = list(layers)
        if len({l.in_features for l in layers}) != 1 or len({l.scaling for l in layers}) != 1:
            raise ValueError("fused projections need the same input size and scaling")
        if not 1 <= len(layers) <= 4:
            raise ValueError("one to four projections per call")
        if any(l.weight is None for l in layers):
            raise ValueError("fused projections need bf16 base weights (not NF4 codes)")
        self.outs = tuple(l.out_features for l in layers)
        self.ranks = tuple(l.r for l in layers)
        if sum(self.ranks) > 64:
            raise ValueError("sum of ranks above 64")
        self.scaling = layers[0].scaling
        self.layers = nn.ModuleList(layers)

    def forward(self, x: torch.Tensor):
        ls = self.layers
        return tuple(_lora_projections(x, [l.weight for l in ls], [l.lora_A for l in ls], [l.lora_B for l in ls],
                                       float(self.scaling), [_frozen_bias(l.bias) for l in ls]))
