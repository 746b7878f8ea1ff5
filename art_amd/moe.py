"""MoE expert block with per-expert LoRA on the MI355X kernels.

Routing (top-k on the router logits, stable expert-contiguous permutation), the
three per-expert projections (gate, up, down; each W_e x + scale B_e A_e x), the
SiLU gating between them and the weighted recombination of a token's k expert
outputs run in the artk library, one call each way.  The reference has no MoE code at this
commit; the shapes follow the Qwen3-30B-A3B-style benchmark configuration."""
from __future__ import annotations

import torch
from torch import nn

from . import ops


def _aligned(t: torch.Tensor) -> torch.Tensor:
    """``t``, contiguous and on the 16 bytes that the library's vector loads need (a view into a flat buffer of
    parameters or gradients may lie anywhere)."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


class _MoEExpertsFn(torch.autograd.Function):
    """The whole block (routing, three projections, gating, recombination) as one library call each way."""

    @staticmethod
    def forward(ctx, x, logits, top_k, W_gu, W_d, Wt_gu, Wt_d, scale, backward, *params):
        dtype = params[0].dtype
        if dtype not in (torch.float32, torch.bfloat16) or any(p.dtype != dtype for p in params):
            dtype = torch.float32
        adapters = {n: _aligned(p.detach().to(dtype)) for n, p in zip(ops._MOE_PARAMS, params)}
        y, routing, saved = ops.moe_experts_fwd(x, logits, top_k, W_gu, W_d, adapters, scale, backward)
        ctx.save_for_backward(x, saved)
        # the module's transposed weights outlive the call: as saved tensors, hooks that move activations to the host
        # would copy them for every block
        ctx.routing, ctx.scale, ctx.frozen = routing, scale, (Wt_gu, Wt_d)
        ctx.rank, ctx.dtypes = params[0].shape[1], [p.dtype for p in params]   # (their values are in `saved`)
        return y, routing

    @staticmethod
    def backward(ctx, g, _g_routing):
        x, saved = ctx.saved_tensors
        dx, grads = ops.moe_experts_bwd(_aligned(g), x, ctx.routing, saved, *ctx.frozen, ctx.rank, ctx.scale)
        return (dx,) + (None,) * 8 + tuple(grads[n].to(t) for n, t in zip(ops._MOE_PARAMS, ctx.dtypes))


class MoELoRAExperts(nn.Module):
    """E experts, each a gated MLP (gate/up [I,H], down [H,I]) with rank-r LoRA."""

    def __init__(self, hidden: int, intermediate: int, n_experts: int, top_k: int, r: int = 8,
                 lora_alpha: int = 16, device=None):
        super().__init__()
        self.top_k, self.scaling = top_k, lora_alpha / r
        bf = dict(device=device, dtype=torch.bfloat16)
        # gate and up read the same rows: they are stored as ONE [E, 2I, H] weight (gate rows first) so
        # that they run as one grouped product (one pass over x, twice the K length in the
        # input-gradient product); `gate_weight` / `up_weight` are views of it, not copies
        self.register_parameter("gate_up_weight", nn.Parameter(
            0.02 * torch.randn(n_experts, 2 * intermediate, hidden, **bf), requires_grad=False))
        self.register_parameter("down_weight", nn.Parameter(
            0.02 * torch.randn(n_experts, hidden, intermediate, **bf), requires_grad=False))
        shapes = {"gate": (intermediate, hidden), "up": (intermediate, hidden), "down": (hidden, intermediate)}
        for name, (o, i) in shapes.items():
            bound = 1.0 / i ** 0.5
            self.register_parameter(f"{name}_lora_A", nn.Parameter(
                (torch.rand(n_experts, r, i, device=device) * 2 - 1) * bound))
            self.register_parameter(f"{name}_lora_B", nn.Parameter(torch.zeros(n_experts, o, r, device=device)))
        self.intermediate = intermediate
        self._wt = {}

    @property
    def gate_weight(self) -> torch.Tensor:
        """[E, I, H] view of the gate rows of gate_up_weight."""
        return self.gate_up_weight[:, :self.intermediate]

    @property
    def up_weight(self) -> torch.Tensor:
        """[E, I, H] view of the up rows of gate_up_weight."""
        return self.gate_up_weight[:, self.intermediate:]

    def _transposed(self, name):
        w = getattr(self, f"{name}_weight")
        hit = self._wt.get(name)
        if hit is None or hit[0] != w._version or hit[1] != w.data_ptr():
            self._wt[name] = (w._version, w.data_ptr(), ops.transpose_batched(w))
        return self._wt[name][2]

    def forward(self, x: torch.Tensor, router_logits: torch.Tensor):
        """x bf16 [T,H], router_logits f32 [T,E] -> (y bf16 [T,H], routing)."""
        params = (self.gate_lora_A, self.gate_lora_B, self.up_lora_A, self.up_lora_B, self.down_lora_A,
                  self.down_lora_B)
        # (inside the function grad mode is off either way)
        backward = torch.is_grad_enabled() and any(t.requires_grad for t in (x, *params))
        return _MoEExpertsFn.apply(
            x.to(torch.bfloat16).contiguous(), router_logits.detach().float().contiguous(), self.top_k,
            self.gate_up_weight, self.down_weight, self._transposed("gate_up"), self._transposed("down"),
            float(self.scaling), backward, *params)
