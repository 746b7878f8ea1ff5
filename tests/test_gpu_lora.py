"""GPU parity of the LoRA linear (forward and backward) against the CPU oracle.

Tolerance: rel-L2 <= 1e-2 for y, dx, dA, dB against the fp32 oracle evaluated
on the same bf16-valued inputs."""
import math
import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import lora_oracle  # noqa: E402

from art_amd import _lib, ops  # noqa: E402
from art_amd.lora import LoRALinear, lora_linear  # noqa: E402

pytestmark = pytest.mark.gpu
TOL = 1e-2


def rel_l2(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


def make(T, n_in, n_out, r, seed, b_std=0.01):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, n_in, generator=g).to(torch.bfloat16)
    W = (0.02 * torch.randn(n_out, n_in, generator=g)).to(torch.bfloat16)
    bound = 1.0 / math.sqrt(n_in)  # Kaiming-uniform with a = sqrt(5)
    A = ((torch.rand(r, n_in, generator=g) * 2 - 1) * bound).to(torch.bfloat16)
    B = (b_std * torch.randn(n_out, r, generator=g)).to(torch.bfloat16)
    up = torch.randn(T, n_out, generator=g).to(torch.bfloat16)
    return x, W, A, B, up


def run_gpu(x, W, A, B, up, scale, gpu):
    xd, Wd, Ad, Bd, upd = (t.to(gpu) for t in (x, W, A, B, up))
    y, xa = ops.lora_linear_fwd(xd, Wd, Ad, Bd, scale)
    dx, dA, dB = ops.lora_linear_bwd(upd, xd, ops.transpose(Wd), Ad, Bd, xa, scale)
    return y.cpu().float(), dx.cpu().float(), dA.cpu(), dB.cpu()


@pytest.mark.parametrize("T,n_in,n_out,r", [(512, 256, 256, 8), (300, 192, 320, 8), (256, 128, 64, 16),
                                            (1000, 512, 576, 24),
                                            (5000, 192, 4160, 8)])  # more tiles than CUs, ragged on both sides
def test_lora_matches_oracle(artk_lib, gpu, T, n_in, n_out, r):
    print(f"lora T={T} in={n_in} out={n_out} r={r}", flush=True)
    x, W, A, B, up = make(T, n_in, n_out, r, T + r)
    scale = 16 / r
    y0, dx0, dA0, dB0 = lora_oracle.lora_linear_grads(x, W, A, B, scale, up)
    y, dx, dA, dB = run_gpu(x, W, A, B, up, scale, gpu)
    assert rel_l2(y, y0) <= TOL
    assert rel_l2(dx, dx0) <= TOL
    assert rel_l2(dA, dA0) <= TOL
    assert rel_l2(dB, dB0) <= TOL


def test_lora_zero_factors(artk_lib, gpu):
    """B = 0: y is the base projection and dA vanishes; A = 0: dB vanishes."""
    x, W, A, B, up = make(256, 128, 192, 8, 5)
    y, dx, dA, dB = run_gpu(x, W, A, torch.zeros_like(B), up, 2.0, gpu)
    base = ops.gemm_nt(W.to(gpu), x.to(gpu)).cpu().float()
    assert torch.equal(y, base)
    assert dA.abs().max().item() == 0.0
    assert dB.abs().max().item() > 0.0
    y, dx, dA, dB = run_gpu(x, W, torch.zeros_like(A), B, up, 2.0, gpu)
    assert dB.abs().max().item() == 0.0
    assert dA.abs().max().item() > 0.0


@pytest.mark.parametrize("n_out", [2048, 256, 11008])
def test_lora_config2_full_size(artk_lib, gpu, n_out):
    """Benchmark config 2 (Qwen2.5-3B projections) at full size."""
    print(f"lora config2 out={n_out}", flush=True)
    x, W, A, B, up = make(8192, 2048, n_out, 8, 1002 + n_out)
    y0, dx0, dA0, dB0 = lora_oracle.lora_linear_grads(x, W, A, B, 2.0, up)
    y, dx, dA, dB = run_gpu(x, W, A, B, up, 2.0, gpu)
    assert rel_l2(y, y0) <= TOL
    assert rel_l2(dx, dx0) <= TOL
    assert rel_l2(dA, dA0) <= TOL
    assert rel_l2(dB, dB0) <= TOL


def test_lora_down_projection_full_size(artk_lib, gpu):
    """The seventh target module of the reference's adapter config (down_proj, 11008 -> 2048,
    src/art/dev/model.py:54-62) at full size, with rank 16."""
    print("lora down_proj 11008 -> 2048, r=16", flush=True)
    x, W, A, B, up = make(4096, 11008, 2048, 16, 1717)
    y0, dx0, dA0, dB0 = lora_oracle.lora_linear_grads(x, W, A, B, 1.0, up)
    y, dx, dA, dB = run_gpu(x, W, A, B, up, 1.0, gpu)
    assert rel_l2(y, y0) <= TOL
    assert rel_l2(dx, dx0) <= TOL
    assert rel_l2(dA, dA0) <= TOL
    assert rel_l2(dB, dB0) <= TOL


def test_lora_module_autograd(artk_lib, gpu):
    torch.manual_seed(0)
    mod = LoRALinear(256, 320, r=8, lora_alpha=16, device=gpu, dtype=torch.float32)
    with torch.no_grad():
        mod.lora_B.normal_(std=0.01)
    x = torch.randn(2, 96, 256, device=gpu, dtype=torch.bfloat16, requires_grad=True)
    y = mod(x)
    assert y.shape == (2, 96, 320)
    up = torch.randn_like(y)
    y.backward(up)
    y0, dx0, dA0, dB0 = lora_oracle.lora_linear_grads(
        x.detach().cpu().view(-1, 256), mod.weight.cpu(), mod.lora_A.detach().cpu().to(torch.bfloat16),
        mod.lora_B.detach().cpu().to(torch.bfloat16), mod.scaling, up.cpu().view(-1, 320))
    assert rel_l2(y.detach().cpu().float().view(-1, 320), y0) <= TOL
    assert rel_l2(x.grad.cpu().float().view(-1, 256), dx0) <= TOL
    assert rel_l2(mod.lora_A.grad.cpu(), dA0) <= TOL
    assert rel_l2(mod.lora_B.grad.cpu(), dB0) <= TOL
    assert mod.weight.grad is None


def test_fused_projections_match_separate(artk_lib, gpu):
    """q/k/v as one product: same outputs and gradients as three LoRALinear modules."""
    from art_amd.lora import FusedLoRALinear, LoRALinear
    torch.manual_seed(5)
    T, n_in = 192, 256
    layers = [LoRALinear(n_in, o, r=8, lora_alpha=16, device=gpu, dtype=torch.float32) for o in (256, 64, 64)]
    for l in layers:
        torch.nn.init.normal_(l.lora_B, std=0.05)
    fused = FusedLoRALinear(layers)
    x1 = torch.randn(T, n_in, device=gpu).to(torch.bfloat16).requires_grad_(True)
    x2 = x1.detach().clone().requires_grad_(True)
    ups = [torch.randn(T, o, device=gpu).to(torch.bfloat16) for o in (256, 64, 64)]
    ys = [l(x1) for l in layers]
    sum((y.float() * u.float()).sum() for y, u in zip(ys, ups)).backward()
    ref = [(l.lora_A.grad.clone(), l.lora_B.grad.clone()) for l in layers]
    for l in layers:
        l.lora_A.grad = None
        l.lora_B.grad = None
    yf = fused(x2)
    sum((y.float() * u.float()).sum() for y, u in zip(yf, ups)).backward()
    rel = lambda a, b: ((a.double() - b.double()).norm() / b.double().norm()).item()
    for a, b in zip(yf, ys):
        assert rel(a.float(), b.float()) <= 4e-3
    assert rel(x2.grad.float(), x1.grad.float()) <= 1e-2
    for l, (dA, dB) in zip(layers, ref):
        assert rel(l.lora_A.grad, dA) <= 1e-2 and rel(l.lora_B.grad, dB) <= 1e-2


@pytest.mark.parametrize("n_out,r", [(2048, 8), (256, 8), (320, 48)])
def test_lora_bias_and_ranks(artk_lib, gpu, n_out, r):
    """Qwen2.5's q/k/v projections carry a (frozen) bias: y = x W^T + bias + s (x A^T) B^T at the
    config-2 q and k/v shapes, and a rank above 32 on a ragged shape (two e tiles in the
    one-pass skinny products).  The bias adds nothing to dx, dA, dB."""
    print(f"lora bias out={n_out} r={r}", flush=True)
    T, n_in = (8192, 2048) if r == 8 else (1100, 448)
    x, W, A, B, up = make(T, n_in, n_out, r, 77 + n_out)
    bias = (0.5 * torch.randn(n_out, generator=torch.Generator().manual_seed(n_out))).to(torch.bfloat16)
    scale = 16 / r
    y0, dx0, dA0, dB0 = lora_oracle.lora_linear_grads(x, W, A, B, scale, up)
    y0 = y0 + bias.float()
    xd, Wd, Ad, Bd, upd = (t.to(gpu) for t in (x, W, A, B, up))
    y, xa = ops.lora_linear_fwd(xd, Wd, Ad, Bd, scale, bias.to(gpu))
    dx, dA, dB = ops.lora_linear_bwd(upd, xd, ops.transpose(Wd), Ad, Bd, xa, scale)
    assert rel_l2(y.cpu().float(), y0) <= TOL
    assert rel_l2(dx.cpu().float(), dx0) <= TOL
    assert rel_l2(dA.cpu(), dA0) <= TOL
    assert rel_l2(dB.cpu(), dB0) <= TOL
    # bit-reproducible run to run (fixed summation orders)
    dx2, dA2, dB2 = ops.lora_linear_bwd(upd, xd, ops.transpose(Wd), Ad, Bd, xa, scale)
    assert torch.equal(dA, dA2) and torch.equal(dB, dB2) and torch.equal(dx, dx2)


def test_lora_module_with_bias_from_linear(artk_lib, gpu):
    """LoRALinear.from_linear keeps the base layer's bias (as peft does) and leaves it frozen."""
    torch.manual_seed(3)
    lin = torch.nn.Linear(256, 192, bias=True, device=gpu, dtype=torch.bfloat16)
    mod = LoRALinear.from_linear(lin, r=8, lora_alpha=16)
    assert mod.bias is not None and not mod.bias.requires_grad
    with torch.no_grad():
        mod.lora_B.normal_(std=0.02)
    x = torch.randn(300, 256, device=gpu, dtype=torch.bfloat16, requires_grad=True)
    y = mod(x)
    y.backward(torch.ones_like(y))
    want = (x.detach().float() @ lin.weight.float().t() + lin.bias.float()
            + mod.scaling * (x.detach().float() @ mod.lora_A.float().t()) @ mod.lora_B.float().t())
    assert rel_l2(y.detach().float().cpu(), want.cpu()) <= TOL
    assert mod.bias.grad is None and mod.lora_A.grad is not None


# ---- projections of the same input in one call (q|k|v, gate|up) ------------------------------------
_oracle_cache = {}


def shared_input_case(T, n_in, outs, ranks, seed, with_bias):
    """Per projection (W, A, B, bias, g) on one x, and the oracle's (y, dx, dA, dB) of each."""
    key = (T, n_in, tuple(outs), tuple(ranks), seed, with_bias)
    if key not in _oracle_cache:
        g = torch.Generator().manual_seed(seed)
        x = torch.randn(T, n_in, generator=g).to(torch.bfloat16)
        parts, refs = [], []
        for o, r in zip(outs, ranks):
            W = (0.02 * torch.randn(o, n_in, generator=g)).to(torch.bfloat16)
            A = ((torch.rand(r, n_in, generator=g) * 2 - 1) / math.sqrt(n_in)).to(torch.bfloat16)
            B = (0.01 * torch.randn(o, r, generator=g)).to(torch.bfloat16)
            bias = (0.5 * torch.randn(o, generator=g)).to(torch.bfloat16) if with_bias else None
            up = torch.randn(T, o, generator=g).to(torch.bfloat16)
            parts.append((W, A, B, bias, up))
        scale = 16 / ranks[0]
        for W, A, B, bias, up in parts:
            y0, dx0, dA0, dB0 = lora_oracle.lora_linear_grads(x, W, A, B, scale, up)
            refs.append((y0 + bias.float() if with_bias else y0, dx0, dA0, dB0))
        _oracle_cache.clear()          # one case at a time: a gate|up case holds 3 GB of fp32 references
        _oracle_cache[key] = (x, parts, refs, scale)
    return _oracle_cache[key]


MULTI_CASES = [
    pytest.param(8192, 2048, (2048, 256, 256), (8, 8, 8), True, id="c2-qkv"),
    pytest.param(8192, 2048, (11008, 11008), (8, 8), False, id="c2-gate_up"),
    pytest.param(300, 192, (320, 64), (16, 16), True, id="ragged"),
    pytest.param(1000, 448, (192, 576, 64, 128), (8, 8, 8, 8), False, id="four"),
]


@pytest.mark.parametrize("T,n_in,outs,ranks,with_bias", MULTI_CASES)
def test_multi_projection_matches_oracle(artk_lib, gpu, T, n_in, outs, ranks, with_bias):
    """artk_lora_linear_multi_fwd / _bwd (separate weights, adapters, outputs and upstream gradients)
    against the oracle evaluated projection by projection; dx is the sum over the projections.  The
    two config-2 cases are the call shapes of a Qwen2.5-3B layer at full size."""
    print(f"lora multi T={T} in={n_in} outs={outs} ranks={ranks}", flush=True)
    x, parts, refs, scale = shared_input_case(T, n_in, outs, ranks, 4242 + T, with_bias)
    xd = x.to(gpu)
    Ws = [p[0].to(gpu) for p in parts]
    As = [p[1].to(gpu) for p in parts]
    Bs = [p[2].to(gpu) for p in parts]
    biases = [p[3].to(gpu) for p in parts] if with_bias else None
    gs = [p[4].to(gpu) for p in parts]
    ys, xas = ops.lora_linear_multi_fwd(xd, Ws, As, Bs, scale, biases)
    dx, dAs, dBs = ops.lora_linear_multi_bwd(gs, xd, [ops.transpose(w) for w in Ws], As, Bs, xas, scale)
    dx0 = sum(r[1] for r in refs)
    assert rel_l2(dx.cpu().float(), dx0) <= TOL
    for i, (y0, _, dA0, dB0) in enumerate(refs):
        assert rel_l2(ys[i].cpu().float(), y0) <= TOL, i
        assert rel_l2(dAs[i].cpu(), dA0) <= TOL, i
        assert rel_l2(dBs[i].cpu(), dB0) <= TOL, i
    # bit-reproducible run to run, and identical to the single-projection entry points on each projection's
    # own outputs (same kernels and summation orders; dx differs: it is one accumulation here)
    dx2, dAs2, dBs2 = ops.lora_linear_multi_bwd(gs, xd, [ops.transpose(w) for w in Ws], As, Bs, xas, scale)
    assert torch.equal(dx, dx2) and all(torch.equal(a, b) for a, b in zip(dAs + dBs, dAs2 + dBs2))
    y_one, xa_one = ops.lora_linear_fwd(xd, Ws[-1], As[-1], Bs[-1], scale, None if biases is None else biases[-1])
    assert torch.equal(y_one, ys[-1]) and torch.equal(xa_one, xas[-1])


@pytest.mark.parametrize("T,n_in,outs,ranks,with_bias", MULTI_CASES[:2])
def test_concatenated_projections_config2_full_size(artk_lib, gpu, T, n_in, outs, ranks, with_bias):
    """The single-projection entry points on the concatenated form of the same cases: weights stacked
    along the output dimension, A stacked, B block-diagonal (out 2560 / rank 24 with the q, k, v biases;
    out 22016 / rank 16).  The diagonal blocks of dB are the adapters' gradients; the off-diagonal
    blocks are derivatives with respect to entries that are pinned to zero and belong to no adapter
    (they are not zero; they are checked against the oracle's full product like the rest)."""
    print(f"lora concatenated out={sum(outs)} r={sum(ranks)}", flush=True)
    x, parts, refs, scale = shared_input_case(T, n_in, outs, ranks, 4242 + T, with_bias)
    W = torch.cat([p[0] for p in parts], 0)
    A = torch.cat([p[1] for p in parts], 0)
    B = torch.zeros(sum(outs), sum(ranks), dtype=torch.bfloat16)
    o0 = r0 = 0
    for (p, o, r) in zip(parts, outs, ranks):
        B[o0:o0 + o, r0:r0 + r] = p[2]
        o0, r0 = o0 + o, r0 + r
    bias = torch.cat([p[3] for p in parts]) if with_bias else None
    up = torch.cat([p[4] for p in parts], 1)
    xd, Wd, Ad, Bd, upd = (t.to(gpu).contiguous() for t in (x, W, A, B, up))
    y, xa = ops.lora_linear_fwd(xd, Wd, Ad, Bd, scale, None if bias is None else bias.to(gpu))
    dx, dA, dB = ops.lora_linear_bwd(upd, xd, ops.transpose(Wd), Ad, Bd, xa, scale)
    assert rel_l2(dx.cpu().float(), sum(r[1] for r in refs)) <= TOL
    o0 = r0 = 0
    for (y0, _, dA0, dB0), o, r in zip(refs, outs, ranks):
        assert rel_l2(y[:, o0:o0 + o].cpu().float(), y0) <= TOL
        assert rel_l2(dA[r0:r0 + r].cpu(), dA0) <= TOL
        assert rel_l2(dB[o0:o0 + o, r0:r0 + r].cpu(), dB0) <= TOL
        o0, r0 = o0 + o, r0 + r
    # the whole dB, off-diagonal blocks included: s g^T (x A_cat^T) in fp64 on the CPU
    xa0 = x.double() @ A.double().t()
    dB_full = scale * (up.double().t() @ xa0)
    assert rel_l2(dB.cpu(), dB_full) <= TOL


@pytest.mark.parametrize("T,n_in,outs,r", [
    (1, 64, (64,), 8),                  # one row, one K step
    (129, 320, (192, 64), 16),          # one row and half a tile past an edge, two jobs
    (130, 4864, (896,), 8),             # long K, few tiles: split in the forward
    (200, 128, (4864, 64), 24),         # input gradient over two segments of very different length, split
    (200, 64, (64, 8192, 128), 8),      # split boundaries inside the middle segment
])
def test_small_products(artk_lib, gpu, T, n_in, outs, r):
    """Sizes that run on 128 x 128 tiles with the K range split: forward with bias and backward of all
    projections against fp32 (1e-2: bf16 outputs and bf16 low-rank products, as for the large tiles)."""
    print("small products", T, n_in, outs, r, flush=True)
    g = torch.Generator().manual_seed(T + n_in)
    rnd = lambda *s, std=1.0: (std * torch.randn(*s, generator=g)).to(torch.bfloat16)
    x = rnd(T, n_in)
    W, A, B = ([rnd(o, n_in, std=0.02) for o in outs], [rnd(r, n_in, std=n_in ** -0.5) for _ in outs],
               [rnd(o, r, std=0.05) for o in outs])
    bias, up = [rnd(o) for o in outs], [rnd(T, o) for o in outs]
    dev = lambda ts: [t.to(gpu) for t in ts]
    ys, xas = ops.lora_linear_multi_fwd(x.to(gpu), dev(W), dev(A), dev(B), 0.5, dev(bias))
    dx, dAs, dBs = ops.lora_linear_multi_bwd(dev(up), x.to(gpu), [ops.transpose(w.to(gpu)) for w in W], dev(A), dev(B),
                                             xas, 0.5)
    rel = lambda a, b: ((a.float().cpu() - b).norm() / b.norm()).item()
    xf, dx0 = x.float(), 0
    for i in range(len(outs)):
        Wf, Af, Bf, gf = (t.float() for t in (W[i], A[i], B[i], up[i]))
        assert rel(ys[i], xf @ Wf.T + bias[i].float() + 0.5 * (xf @ Af.T) @ Bf.T) <= 1e-2
        assert rel(dAs[i], 0.5 * (gf @ Bf).T @ xf) <= 1e-2 and rel(dBs[i], 0.5 * gf.T @ (xf @ Af.T)) <= 1e-2
        dx0 = dx0 + gf @ Wf + 0.5 * (gf @ Bf) @ Af
        y1, _ = ops.lora_linear_fwd(x.to(gpu), W[i].to(gpu), A[i].to(gpu), B[i].to(gpu), 0.5, bias[i].to(gpu))
        assert rel(y1, ys[i].float().cpu()) <= 4e-3   # one rounding to bf16; the K range may be split elsewhere
    assert rel(dx, dx0) <= 1e-2


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_native_autograd_function(artk_lib, gpu, dtype):
    """The native autograd function around the projections: leading dimensions, an fp32 input, adapters in either
    dtype (gradients come back in it), an output nobody uses, no graph under no_grad, and an in-place change of
    the frozen weight between forward and backward, which is an error.  1e-2: bf16 products; the gradients of
    bf16 adapters are the fp32 sums rounded once (4e-3)."""
    from art_amd.lora import FusedLoRALinear, LoRALinear

    torch.manual_seed(5)
    T, n_in, outs, r = 70, 128, (192, 64), 8
    layers = [LoRALinear(n_in, o, r=r, lora_alpha=16, device=gpu, dtype=dtype) for o in outs]
    with torch.no_grad():
        for l in layers:
            l.lora_B.normal_(std=0.05)
    mod = FusedLoRALinear(layers)
    x = torch.randn(2, T // 2, n_in, device=gpu, requires_grad=True)
    up = torch.randn(2, T // 2, outs[0], device=gpu)
    y, _ = mod(x)
    assert y.shape == (2, T // 2, outs[0]) and y.dtype == torch.bfloat16
    y.backward(up.to(torch.bfloat16))
    f = lambda t: t.detach().to(torch.bfloat16).float().cpu()
    xf, gf, W, A, B = f(x).view(T, n_in), f(up).view(T, outs[0]), f(layers[0].weight), f(layers[0].lora_A), f(layers[0].lora_B)
    rel = lambda a, b: ((a.float().cpu() - b).norm() / b.norm()).item()
    assert x.grad.dtype == torch.float32 and rel(x.grad.view(T, n_in), gf @ W + 2.0 * (gf @ B) @ A) <= 1e-2
    assert layers[0].lora_A.grad.dtype == dtype and rel(layers[0].lora_A.grad, 2.0 * (gf @ B).T @ xf) <= 1e-2
    assert layers[0].lora_B.grad.dtype == dtype and rel(layers[0].lora_B.grad, 2.0 * gf.T @ (xf @ A.T)) <= 1e-2
    assert layers[1].lora_A.grad.abs().max().item() == 0.0 and layers[1].lora_B.grad.abs().max().item() == 0.0
    with torch.no_grad():
        y2, _ = mod(x)
    assert not y2.requires_grad and torch.equal(y2, y)
    y3, _ = mod(x)
    with torch.no_grad():
        layers[0].weight.mul_(2.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y3.sum().backward()
    with pytest.raises(ValueError):
        mod(x.cpu())


def test_saved_tensor_hooks_see_activations_only(artk_lib, gpu):
    """Hooks that move saved tensors to the host (torch.autograd.graph.save_on_cpu) see the activations, adapters
    and frozen bf16 weights, not the 4-bit codes, the transposed weights or the attention plan, which outlive the
    call anyway; the gradients are the same bits."""
    from art_amd import attention, quant
    from art_amd.lora import LoRALinear

    torch.manual_seed(6)
    dense = LoRALinear(128, 192, device=gpu)
    nf4 = LoRALinear.from_nf4(quant.NF4Weight.from_float(torch.randn(64, 192, device=gpu).to(torch.bfloat16)))
    ids = torch.zeros(1, 70, dtype=torch.int64, device=gpu)
    plans = attention.attention_plans(ids, ids)
    x = torch.randn(1, 70, 128, device=gpu, dtype=torch.bfloat16, requires_grad=True)

    def step():
        h = dense(x)
        q = h.view(1, 70, 3, 64)
        y = nf4(attention.packed_attention(q, q[:, :, :1], q[:, :, 1:2], plans).reshape(1, 70, 192))
        return torch.autograd.grad(y.float().sum(), [x, dense.lora_A, nf4.lora_B])

    want = step()
    seen = []

    def pack(t):
        seen.append((t.dtype, tuple(t.shape)))
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(gpu)):
        got = step()
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert (torch.bfloat16, (192, 128)) in seen and (torch.bfloat16, (128, 192)) not in seen
    assert not any(dtype == torch.uint8 for dtype, _ in seen)


def test_native_functions_on_another_stream(artk_lib, gpu):
    """The projections and packed attention, forward and backward, on a stream that is not the default one while the
    default stream is busy: inputs made on that stream, the bits of the default stream's results."""
    from art_amd import attention
    from art_amd.lora import FusedLoRALinear, LoRALinear

    torch.manual_seed(8)
    layers = [LoRALinear(256, o, device=gpu) for o in (256, 64, 64)]
    for m in layers:
        m.lora_B.data.normal_(std=0.05)
    fused = FusedLoRALinear(layers)
    ids = torch.zeros(2, 300, dtype=torch.int64, device=gpu)
    host = torch.randn(2, 300, 256, dtype=torch.bfloat16)
    params = [p for m in layers for p in (m.lora_A, m.lora_B)]

    def step(x):
        x = x.detach().requires_grad_(True)
        q, k, v = (t.view(2, 300, -1, 64) for t in fused(x))
        out = attention.packed_attention(q, k, v, attention.attention_plans(ids, ids))
        return [out.detach(), *torch.autograd.grad(out.float().square().sum(), [x] + params)]

    want = step(host.to(gpu))
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    busy = torch.randn(4096, 4096, device=gpu)
    for _ in range(20):
        busy = busy @ busy * 1e-3
    with torch.cuda.stream(side):
        got = step(host.to(gpu, non_blocking=True))
    side.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_forward_makes_no_transposed_weight(artk_lib, gpu):
    """A forward with a graph but without a backward keeps no second copy of a weight; the first backward makes it, of
    the module's own weight also where saved-tensor hooks hand the node a copy, and the gradients are those of later
    passes, in which the copy is there."""
    from art_amd.lora import FusedLoRALinear, LoRALinear

    torch.manual_seed(9)
    layers = [LoRALinear(128, o, device=gpu) for o in (192, 64)]
    for m in layers:
        m.lora_B.data.normal_(std=0.05)
    fused = FusedLoRALinear(layers)
    x = torch.randn(1, 70, 128, device=gpu, dtype=torch.bfloat16, requires_grad=True)
    params = [p for m in layers for p in (m.lora_A, m.lora_B)]

    def grads():
        return torch.autograd.grad(sum(y.float().square().sum() for y in fused(x)), [x] + params)

    fused(x)
    assert all(ops.known_transpose(m.weight) is None for m in layers)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(gpu)):
        first = grads()
    assert all(torch.equal(ops.known_transpose(m.weight), m.weight.t()) for m in layers)
    for a, b in zip(first, grads()):
        assert torch.equal(a, b)
    with torch.no_grad():
        layers[0].weight.mul_(2)
    assert ops.known_transpose(layers[0].weight) is None
    for a, b in zip(grads(), grads()):
        assert torch.equal(a, b)


@pytest.mark.parametrize("T,n_in,n_out,r", [
    (1, 64, 64, 8), (63, 128, 192, 16), (65, 640, 448, 8),        # one row, around a 64-row tile, ragged 128-column tiles
    (257, 64, 576, 16),                                           # one column tile: the ring runs over row tiles alone
    (129, 4160, 1088, 8),                                         # several chunks of columns
    (8192, 64, 16448, 16),                                        # more than 256 MiB of g: non-temporal loads
    (65, 640, 448, 24), (1, 128, 64, 32), (300, 64, 1088, 32),    # two blocks of 16 ranks
    (130, 192, 448, 40)])                                         # the kernel of larger ranks
def test_skinny_passes_of_small_ranks(artk_lib, gpu, T, n_in, n_out, r):
    """dA, dB and, through dx, g B at the edges of the one-pass backward.  TOL as above: bf16 factors
    on the way."""
    print(f"skinny passes T={T} in={n_in} out={n_out} r={r}", flush=True)
    x, W, A, B, up = (t.to(gpu) for t in make(T, n_in, n_out, r, T + n_out, b_std=0.3))
    scale = 2.0
    _, xa = ops.lora_linear_fwd(x, W, A, B, scale)
    dx, dA, dB = ops.lora_linear_bwd(up, x, ops.transpose(W), A, B, xa, scale)
    # an infinity in the last row and column reaches its own sums only
    up2, x2 = up.clone(), x.clone()
    up2[-1, -1] = float("inf")
    x2[-1, -1] = float("inf")
    _, dA2, dB2 = ops.lora_linear_bwd(up2, x2, ops.transpose(W), A, B, xa.clamp(min=0.5), scale)
    assert torch.isfinite(dB2[:-1]).all() and torch.isinf(dB2[-1]).all()
    assert torch.isfinite(dA2[:, :-1]).sum() == 0
    g, xf, Af, Bf = up.float(), x.float(), A.float(), B.float()
    gb = g @ Bf
    assert rel_l2(dA, scale * gb.t() @ xf) <= TOL
    assert rel_l2(dB, scale * g.t() @ (xf @ Af.t())) <= TOL
    assert rel_l2(dx, g @ W.float() + scale * gb @ Af) <= TOL


@pytest.mark.parametrize("T,n_in,ranks", [
    (4097, 64, (8, 24, 16, 40)),      # packed: blocks of 16 factor rows over several ranks, 6 of them
    (4100, 1600, (8, 8, 8)),          # packed, the last pieces of K short
    (5000, 192, (64, 64, 64, 64)),
    (4100, 192, (24,)), (4097, 640, (40,)),  # one factor of several blocks, packed
    (37, 448, (8, 16)),               # few rows: every factor starts its own block
    (37, 8256, (16,)), (2000, 8192, (8,)),  # long K over few rows: split over the chunks of the one-pass kernel
])
def test_row_products(artk_lib, gpu, T, n_in, ranks):
    """x A_i^T of every way the row products are dealt out, element by element: fp32 sums of bf16 products, of which none
    here has more than 34 MFMA steps and additions of partial sums (K / 128 steps and four waves; 16 steps and the chunks
    of the split form), each off by at most 2^-24 of sum |x a|: 2e-6 of it."""
    print(f"row products T={T} in={n_in} ranks={ranks}", flush=True)
    g = torch.Generator().manual_seed(T + n_in)
    x = torch.randn(T, n_in, generator=g).to(torch.bfloat16).to(gpu)
    x[0, :4] = float("inf")            # reaches its own row only
    rand = lambda *s: (0.1 * torch.randn(*s, generator=g)).to(torch.bfloat16).to(gpu)
    Ws, As, Bs = [rand(64, n_in) for _ in ranks], [rand(r, n_in) for r in ranks], [rand(64, r) for r in ranks]
    for A in As:
        A[:, :4] = A[:, :4].abs() + 0.1
    _, xas = ops.lora_linear_multi_fwd(x, Ws, As, Bs, 2.0)
    for A, xa in zip(As, xas):
        assert torch.isinf(xa[0]).all()
        ref = x[1:].double() @ A.double().t()
        bound = x[1:].double().abs() @ A.double().abs().t()
        assert ((xa[1:].double() - ref).abs() <= 2e-6 * bound).all()


def partial_units(T, K, Ms):
    """Units of 256 x 256 fp32 partial sums in the workspace of products [M_i, K] x [T, K]^T (at rank 24, where nothing else
    in it comes near one)."""
    proj = (_lib.LoraProjStruct * len(Ms))()
    for p, M in zip(proj, Ms):
        p.out, p.r = M, 24
    return _lib.load().artk_lora_linear_multi_fwd_workspace_bytes(T, K, proj, len(Ms)) // (256 * 256 * 4)


@pytest.mark.parametrize("T,n_in,outs,way", [
    (1500, 11008, (2048,), "forward"),               # rows that are no multiple of a tile
    (1000, 16384, (960, 1088), "forward"),           # two jobs, ragged weight tiles
    (700, 18944, (1088, 1088, 1088), "forward"),     # three
    (1300, 2048, (11008, 11008), "backward"),        # input gradient: parts that span both projections
    (1300, 1984, (11008, 11072), "backward"),        # and ragged weight tiles
])
def test_long_products_of_few_tiles(artk_lib, gpu, T, n_in, outs, way):
    """Products whose K range is split over work-groups on 256 x 256 tiles, block by block (bf16 output rounding: 2e-3
    relative; a part that is missing or added twice is an eighth of the block or more)."""
    K, Ms = (n_in, outs) if way == "forward" else (sum(outs), (n_in,))
    tiles = sum((M + 255) // 256 for M in Ms) * ((T + 255) // 256)
    units = partial_units(T, K, Ms)
    assert units % tiles == 0 and 2 <= units // tiles <= 8, "the shape runs on other tiles now: choose another"
    print(f"long products T={T} in={n_in} outs={outs}", flush=True)
    g = torch.Generator().manual_seed(T)
    rand = lambda *s, std=1.0: (std * torch.randn(*s, generator=g)).to(torch.bfloat16).to(gpu)
    x, r = rand(T, n_in), 8
    Ws, As = [rand(o, n_in, std=0.02) for o in outs], [rand(r, n_in, std=0.02) for _ in outs]
    Bs, ups, biases = [rand(o, r, std=0.2) for o in outs], [rand(T, o) for o in outs], [rand(o, std=0.5) for o in outs]
    ys, xas = ops.lora_linear_multi_fwd(x, Ws, As, Bs, 2.0, biases)
    dx, _, _ = ops.lora_linear_multi_bwd(ups, x, [ops.transpose(w) for w in Ws], As, Bs, xas, 2.0)
    pairs = [(y, x.float() @ W.float().t() + 2.0 * (x.float() @ A.float().t()) @ B.float().t() + b.float())
             for y, W, A, B, b in zip(ys, Ws, As, Bs, biases)]
    pairs.append((dx, sum(u.float() @ W.float() + 2.0 * (u.float() @ B.float()) @ A.float()
                          for u, W, A, B in zip(ups, Ws, As, Bs))))
    for a, ref in pairs:
        for i in range(0, a.shape[0], 32):
            for j in range(0, a.shape[1], 512):
                assert rel_l2(a[i:i + 32, j:j + 512].float(), ref[i:i + 32, j:j + 512]) <= TOL, (i, j)
