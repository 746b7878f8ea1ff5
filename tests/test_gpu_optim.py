"""GPU parity of the fused AdamW step against torch.optim.AdamW + clip_grad_norm_
on the CPU (fp32).  Tolerance 2e-6 relative on parameters and moments after five
steps: the update is the same fp32 arithmetic up to the order of a few roundings."""
import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import optim_oracle  # noqa: E402

from art_amd import ops  # noqa: E402
from art_amd.optim import FlatParams, FusedAdamW  # noqa: E402

pytestmark = pytest.mark.gpu


def rel(a, b):
    return ((a.double() - b.double()).abs().max() / b.double().abs().max()).item()


@pytest.mark.parametrize("n", [1, 7, 4096, 1_000_003])
def test_sumsq(artk_lib, gpu, n):
    x = torch.randn(n, generator=torch.Generator().manual_seed(n))
    got = ops.sumsq(x.to(gpu)).item()
    want = x.double().pow(2).sum().item()
    assert abs(got - want) <= 1e-6 * want
    assert ops.sumsq(x.to(gpu)).item() == got  # fixed order


@pytest.mark.parametrize("clip", [0.1, 0.0])
@pytest.mark.parametrize("lr,wd", [(5e-6, 0.1), (1e-2, 0.0)])
def test_adamw_matches_torch(artk_lib, gpu, clip, lr, wd):
    g = torch.Generator().manual_seed(3)
    shapes = {"A0": (8, 100), "B0": (100, 8), "A1": (8, 37), "B1": (37, 8), "odd": (13,)}
    flat = FlatParams(shapes, gpu)
    flat.master.copy_(torch.randn(flat.numel, generator=g) * 0.05)
    p0 = flat.master.cpu().clone()
    grads = [torch.randn(flat.numel, generator=g) * (0.5 if i % 2 else 0.01) for i in range(5)]
    opt = FusedAdamW(flat, lr=lr, betas=(0.9, 0.99), eps=1e-8, weight_decay=wd, max_grad_norm=clip)
    norms = []
    for gr in grads:
        flat.grad.copy_(gr)
        norms.append(opt.step().item())
    ref_p, ref_m, ref_v, ref_norms = optim_oracle.adamw_steps(p0, grads, lr, (0.9, 0.99), 1e-8, wd, clip)
    for a, b in zip(norms, ref_norms):
        assert abs(a - b) <= 1e-5 * b
    assert rel(flat.master.cpu(), ref_p) <= 2e-6
    assert rel(opt.exp_avg.cpu(), ref_m) <= 2e-6
    assert rel(opt.exp_avg_sq.cpu(), ref_v) <= 2e-6
    # the bf16 copy is the rounded master copy, and the named views alias the flat buffers
    assert torch.equal(flat.shadow, flat.master.to(torch.bfloat16))
    assert flat.param("B1").data_ptr() == flat.master.data_ptr() + 4 * flat.offsets["B1"][0]
    assert flat.bf16("A1").shape == (8, 37)


def test_adamw8bit_matches_oracle(artk_lib, gpu):
    """8-bit block-wise moments: five steps against the numpy restatement.  The arithmetic is the
    same float32 operations; the compiler may fuse a multiply-add, so a value that sits on the
    boundary between two codes can fall on the other side: codes must agree on 99.9 % of the
    elements and never differ by more than one, parameters to 1e-6 relative."""
    import numpy as np

    from art_amd.optim import FusedAdamW8bit, dynamic_code_book

    print("adamw 8-bit", flush=True)
    g = torch.Generator().manual_seed(13)
    shapes = {"A0": (8, 2048), "B0": (2048, 8), "A1": (8, 37), "odd": (13,)}
    flat = FlatParams(shapes, gpu)
    flat.master.copy_(torch.randn(flat.numel, generator=g) * 0.05)
    n = flat.numel
    p = flat.master.cpu().numpy().copy()
    grads = [torch.randn(n, generator=g) * (0.5 if i % 2 else 0.01) for i in range(5)]
    lr, wd, eps, betas, clip = 1e-3, 0.1, 1e-8, (0.9, 0.99), 0.1
    opt = FusedAdamW8bit(flat, lr=lr, betas=betas, eps=eps, weight_decay=wd, max_grad_norm=clip)
    b1, b2 = dynamic_code_book(True).numpy(), dynamic_code_book(False).numpy()
    nb = (n + 255) // 256
    c1 = c2 = np.zeros(n, np.uint8)
    a1 = a2 = np.zeros(nb, np.float32)
    for t, gr in enumerate(grads, 1):
        flat.grad.copy_(gr)
        opt.step()
        p, c1, c2, a1, a2 = optim_oracle.adamw8bit_step(p, gr.numpy(), c1, c2, a1, a2, b1, b2, lr, betas, eps,
                                                        wd, t, clip)
        # continue the oracle from the kernel's own stored state, so that one flipped code
        # does not compound over the steps
        got1, got2 = opt.state1.cpu().numpy(), opt.state2.cpu().numpy()
        d1 = np.abs(got1.astype(int) - c1.astype(int))
        d2 = np.abs(got2.astype(int) - c2.astype(int))
        assert (d1 == 0).mean() >= 0.999 and (d2 == 0).mean() >= 0.999 and d1.max() <= 1 and d2.max() <= 1, t
        assert np.allclose(opt.absmax1.cpu().numpy(), a1, rtol=2e-6, atol=0)
        assert np.allclose(opt.absmax2.cpu().numpy(), a2, rtol=2e-6, atol=0)
        got_p = flat.master.cpu().numpy()
        assert np.abs(got_p - p).max() <= 1e-6 * np.abs(p).max(), t
        c1, c2, a1, a2, p = got1, got2, opt.absmax1.cpu().numpy(), opt.absmax2.cpu().numpy(), got_p
    assert torch.equal(flat.shadow, flat.master.to(torch.bfloat16))
    assert opt.exp_avg().shape == (n,) and opt.exp_avg_sq().min().item() >= 0.0


@pytest.mark.parametrize("n", [5, 256 * 3 + 17, 256 * 16 * 512 + 300])
@pytest.mark.parametrize("book", ["dynamic", "linear", "clustered", "gap"])
def test_adamw8bit_any_code_book(artk_lib, gpu, n, book):
    """One step from a given state at the edges of the grid (less than one block, a last partial block, more
    blocks than waves) and for code books whose entries crowd a bin of the start table or leave most of them
    empty.  Same bounds as test_adamw8bit_matches_oracle, for the same reason."""
    import numpy as np

    from art_amd.optim import dynamic_code_book

    print("adamw 8-bit", n, book, flush=True)
    rng = np.random.default_rng(n)
    if book == "dynamic":
        b1, b2 = dynamic_code_book(True).numpy(), dynamic_code_book(False).numpy()
    elif book == "linear":
        b1, b2 = np.linspace(-1, 1, 256, dtype=np.float32), np.linspace(0, 1, 256, dtype=np.float32)
    elif book == "gap":
        b1 = np.linspace(-1, 1, 256, dtype=np.float32)
        b1[:128], b1[128:] = -np.linspace(1, 0.25, 128), np.linspace(0.25, 1, 128)
        b2 = np.linspace(0.25, 1, 256, dtype=np.float32)
    else:
        b1 = np.sort(np.concatenate([[-1, 0, 1], 0.5 + 1e-3 * rng.random(253)])).astype(np.float32)
        b2 = np.sort(np.concatenate([[0, 1], 1e-8 * rng.random(100), 0.7 + 1e-2 * rng.random(154)])).astype(np.float32)
    nb = (n + 255) // 256
    p = (0.05 * rng.standard_normal(n)).astype(np.float32)
    g = (0.01 * rng.standard_normal(n)).astype(np.float32)
    c1, c2 = rng.integers(0, 256, n).astype(np.uint8), rng.integers(0, 256, n).astype(np.uint8)
    a1, a2 = (1e-3 * rng.random(nb)).astype(np.float32), (1e-6 * rng.random(nb)).astype(np.float32)
    want = optim_oracle.adamw8bit_step(p, g, c1, c2, a1, a2, b1, b2, 1e-3, (0.9, 0.99), 1e-8, 0.1, 3, 0.0)
    t = [torch.from_numpy(x.copy()).to(gpu) for x in (p, g, c1, c2, a1, a2, b1, b2)]
    shadow = torch.zeros(n, dtype=torch.bfloat16, device=gpu)
    ops.adamw8bit_step(*t, shadow, 1e-3, 0.9, 0.99, 1e-8, 0.1, 3)
    for got, ref in ((t[2], want[1]), (t[3], want[2])):
        d = np.abs(got.cpu().numpy().astype(int) - ref.astype(int))
        assert (d == 0).mean() >= 0.999 and d.max() <= 1
    assert np.allclose(t[4].cpu().numpy(), want[3], rtol=2e-6, atol=0)
    assert np.allclose(t[5].cpu().numpy(), want[4], rtol=2e-6, atol=0)
    assert np.abs(t[0].cpu().numpy() - want[0]).max() <= 1e-6 * np.abs(want[0]).max()
    assert torch.equal(shadow, t[0].to(torch.bfloat16))


@pytest.mark.parametrize("exponents", [(-140, -100), (-66, -54), (54, 90)])
def test_adamw8bit_block_maxima_of_any_size(artk_lib, gpu, exponents):
    """Re-quantisation of moments whose block maxima are zero, subnormal, small or large: the quotient by the
    maximum is taken with a scaled reciprocal.  The gradients are zero, so that the moments stay what the codes and block maxima say, times beta;
    same bounds as test_adamw8bit_any_code_book."""
    import numpy as np

    from art_amd.optim import dynamic_code_book

    print("adamw 8-bit maxima", exponents, flush=True)
    n = 256 * 64 + 9
    rng = np.random.default_rng(7)
    nb = (n + 255) // 256
    b1, b2 = dynamic_code_book(True).numpy(), dynamic_code_book(False).numpy()
    p, g = np.zeros(n, np.float32), np.zeros(n, np.float32)
    c1, c2 = rng.integers(0, 256, n).astype(np.uint8), rng.integers(0, 256, n).astype(np.uint8)
    a1, a2 = (np.exp2(rng.uniform(*exponents, nb)).astype(np.float32) for _ in range(2))
    a1[3] = a2[5] = 0.0
    want = optim_oracle.adamw8bit_step(p, g, c1, c2, a1, a2, b1, b2, 0.0, (0.9, 0.99), 1e-8, 0.0, 3, 0.0)
    t = [torch.from_numpy(x.copy()).to(gpu) for x in (p, g, c1, c2, a1, a2, b1, b2)]
    shadow = torch.zeros(n, dtype=torch.bfloat16, device=gpu)
    ops.adamw8bit_step(*t, shadow, 0.0, 0.9, 0.99, 1e-8, 0.0, 3)
    for got, ref in ((t[2], want[1]), (t[3], want[2])):
        d = np.abs(got.cpu().numpy().astype(int) - ref.astype(int))
        assert (d == 0).mean() >= 0.999 and d.max() <= 1
    assert np.allclose(t[4].cpu().numpy(), want[3], rtol=2e-6, atol=0)
    assert np.allclose(t[5].cpu().numpy(), want[4], rtol=2e-6, atol=0)


def test_adamw8bit_non_finite_gradients(artk_lib, gpu):
    """Codes and block maxima where gradients are not finite (fresh moments): a block of NaN keeps NaN as its maximum and
    the code of 0; NaN among zeros leaves a maximum of 0 and codes of 0; NaN and infinities among numbers get code 1, and
    next to an infinity a finite element is 0."""
    import numpy as np

    from art_amd.optim import dynamic_code_book

    print("adamw 8-bit non-finite", flush=True)
    books = [dynamic_code_book(s).numpy() for s in (True, False)]
    zero = [int(optim_oracle.nearest_code(b, np.zeros(1, np.float32))[0]) for b in books]
    n = 4 * 256 + 17
    g = np.zeros(n, np.float32)
    g[:256] = g[4 * 256:] = np.nan      # a whole block, and a last block that is not full
    g[[256 + 3, 256 + 70, 511]] = np.nan
    g[512:1024] = 0.01
    g[512 + 5] = np.inf
    g[768 + 7] = np.nan
    t = [torch.zeros(n, device=gpu), torch.from_numpy(g).to(gpu)]
    t += [torch.full((n,), z, dtype=torch.uint8, device=gpu) for z in zero] + [torch.zeros(5, device=gpu) for _ in range(2)]
    t += [torch.from_numpy(b).to(gpu) for b in books]
    ops.adamw8bit_step(*t, torch.zeros(n, dtype=torch.bfloat16, device=gpu), 1e-3, 0.9, 0.99, 1e-8, 0.0, 1)
    for codes, maxima, z, one in zip(t[2:4], t[4:6], zero, (np.float32(1e-3), np.float32(1e-6))):
        c, a = codes.cpu().numpy(), maxima.cpu().numpy()
        want = np.full(n, z)
        want[768:1024] = 255
        want[[512 + 5, 768 + 7]] = 1
        assert (c == want).all()
        assert np.isnan(a[0]) and a[1] == 0 and np.isinf(a[2]) and np.isclose(a[3], one, rtol=1e-5) and a[4] == 0


@pytest.mark.parametrize("moments", ["8 bit", "fp32"])
def test_steps_past_the_cache_match_steps_of_parts(artk_lib, gpu, moments):
    """A step over more than the caches hold reads and writes past them: bit for bit the steps of its parts."""
    from art_amd.optim import dynamic_code_book

    n = 256 * 74000  # 18.9 M: above both limits, the parts below
    print("adamw past the cache", moments, n, flush=True)
    gen = torch.Generator(device=gpu).manual_seed(3)
    rand = lambda s: torch.randn(n, generator=gen, device=gpu) * s
    p, g = rand(0.05), rand(0.01)
    parts = [slice(0, 256 * 30000), slice(256 * 30000, n)]
    if moments == "fp32":
        m, v = rand(1e-3), rand(1e-3).abs()
        state = [p, g, m, v, torch.zeros(n, dtype=torch.bfloat16, device=gpu)]
        step = lambda t: ops.adamw_step(*t, 1e-3, 0.9, 0.99, 1e-8, 0.1, 3)
        cut = lambda s: [t[s].clone() for t in state]
    else:
        c = [torch.randint(0, 256, (n,), generator=gen, device=gpu).to(torch.uint8) for _ in range(2)]
        a = [torch.rand(n // 256, generator=gen, device=gpu) * x for x in (1e-3, 1e-6)]
        books = [dynamic_code_book(True).to(gpu), dynamic_code_book(False).to(gpu)]
        state = [p, g, *c, *a, *books, torch.zeros(n, dtype=torch.bfloat16, device=gpu)]
        step = lambda t: ops.adamw8bit_step(*t, 1e-3, 0.9, 0.99, 1e-8, 0.1, 3)
        at = lambda t, s: t if t.numel() == 256 else t[slice(s.start // 256, s.stop // 256)] if t.numel() < n else t[s]
        cut = lambda s: [at(t, s).clone() for t in state]
    small = [cut(s) for s in parts]
    for t in small:
        step(t)
    step(state)
    for i, t in enumerate(state):
        if t.numel() != 256:
            assert torch.equal(t, torch.cat([x[i] for x in small])), i
