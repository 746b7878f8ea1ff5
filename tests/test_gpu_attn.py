"""GPU parity of the packed-row attention against the CPU oracle.

Tolerances (fp32 oracle on the bf16-valued inputs): out <= 2e-2 abs on O(1)
values and <= 1e-2 rel-L2, lse <= 2e-3 abs; the equality codes of the plan are
integer work and must reproduce the id equalities exactly.
"""
import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import attn_oracle  # noqa: E402

from art_amd import ops, synthetic  # noqa: E402

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


def make_qkv(seed, S, Hq, Hkv, D):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(S, Hq, D, generator=g).to(torch.bfloat16)
    k = torch.randn(S, Hkv, D, generator=g).to(torch.bfloat16)
    v = torch.randn(S, Hkv, D, generator=g).to(torch.bfloat16)
    return q, k, v


LAYOUTS = {
    # name: (S, n_prompts, prompt_len, n_completions, completion_len)
    "two_prompts": (512, 2, 40, 3, 70),
    "one_long": (512, 1, 100, 1, 412),
    "many_short": (768, 6, 16, 4, 27),
    "no_pad": (256, 1, 64, 3, 64),
}


@pytest.mark.parametrize("layout", list(LAYOUTS))
def test_plan_codes_reproduce_id_equalities(artk_lib, gpu, layout):
    S, npr, pl, nc, cl = LAYOUTS[layout]
    group, parent = synthetic.packed_row_ids(7, S, npr, pl, nc, cl)
    plan = ops.attn_plan(group.to(gpu), parent.to(gpu))
    codes = plan.buf.cpu()
    gc = codes[:4 * S].view(torch.int32)
    off = (4 * S + 255) // 256 * 256
    pc = codes[off:off + 4 * S].view(torch.int32)
    assert torch.equal(gc.unsqueeze(1) == gc.unsqueeze(0), group.unsqueeze(1) == group.unsqueeze(0))
    assert torch.equal(pc.unsqueeze(1) == gc.unsqueeze(0), parent.unsqueeze(1) == group.unsqueeze(0))


@pytest.mark.parametrize("layout", list(LAYOUTS))
@pytest.mark.parametrize("Hq,Hkv,D", [(4, 2, 128), (2, 2, 64), (7, 1, 128)])
def test_attn_fwd_matches_oracle(artk_lib, gpu, layout, Hq, Hkv, D):
    S, npr, pl, nc, cl = LAYOUTS[layout]
    print(f"attn fwd {layout} Hq={Hq} Hkv={Hkv} D={D}", flush=True)
    q, k, v = make_qkv(S + Hq + D, S, Hq, Hkv, D)
    group, parent = synthetic.packed_row_ids(S, S, npr, pl, nc, cl)
    ref_out, ref_lse = attn_oracle.attention(q, k, v, group, parent)
    plan = ops.attn_plan(group.to(gpu), parent.to(gpu))
    out, lse = ops.attn_fwd(q.to(gpu), k.to(gpu), v.to(gpu), plan)
    assert (lse.cpu() - ref_lse).abs().max().item() <= 2e-3
    assert (out.float().cpu() - ref_out).abs().max().item() <= 2e-2
    assert rel_l2(out.float().cpu(), ref_out) <= 1e-2


def test_attn_fwd_head_major_layout_and_random_ids(artk_lib, gpu):
    """[H, S, D] storage (strided views) and ids that are not laid out in
    contiguous segments: the rule is evaluated per element."""
    S, Hq, Hkv, D = 512, 4, 2, 128
    q, k, v = make_qkv(11, S, Hq, Hkv, D)
    g = torch.Generator().manual_seed(12)
    group = torch.randint(0, 5, (S,), generator=g)
    parent = torch.randint(0, 5, (S,), generator=g)
    ref_out, ref_lse = attn_oracle.attention(q, k, v, group, parent)
    plan = ops.attn_plan(group.to(gpu), parent.to(gpu))
    hm = lambda t: t.to(gpu).permute(1, 0, 2).contiguous().permute(1, 0, 2)  # [S,H,D] view of [H,S,D]
    out, lse = ops.attn_fwd(hm(q), hm(k), hm(v), plan)
    assert (lse.cpu() - ref_lse).abs().max().item() <= 2e-3
    assert rel_l2(out.float().cpu(), ref_out) <= 1e-2


@pytest.mark.parametrize("layout", list(LAYOUTS))
@pytest.mark.parametrize("Hq,Hkv,D", [(4, 2, 128), (2, 2, 64), (7, 1, 128)])
def test_attn_bwd_matches_oracle(artk_lib, gpu, layout, Hq, Hkv, D):
    S, npr, pl, nc, cl = LAYOUTS[layout]
    print(f"attn bwd {layout} Hq={Hq} Hkv={Hkv} D={D}", flush=True)
    q, k, v = make_qkv(S + Hq + D + 1, S, Hq, Hkv, D)
    g = torch.Generator().manual_seed(S + 5)
    d_out = torch.randn(S, Hq, D, generator=g).to(torch.bfloat16)
    group, parent = synthetic.packed_row_ids(S + 1, S, npr, pl, nc, cl)
    _, ref_dq, ref_dk, ref_dv = attn_oracle.attention_grads(q, k, v, group, parent, d_out)
    plan = ops.attn_plan(group.to(gpu), parent.to(gpu))
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    out, lse = ops.attn_fwd(qd, kd, vd, plan)
    dq, dk, dv = ops.attn_bwd(qd, kd, vd, out, lse, d_out.to(gpu), plan)
    assert rel_l2(dv.float().cpu(), ref_dv) <= 1e-2
    assert rel_l2(dq.float().cpu(), ref_dq) <= 1e-2
    assert rel_l2(dk.float().cpu(), ref_dk) <= 1e-2
    # run-to-run determinism (no atomics)
    dq2, dk2, dv2 = ops.attn_bwd(qd, kd, vd, out, lse, d_out.to(gpu), plan)
    assert torch.equal(dq, dq2) and torch.equal(dk, dk2) and torch.equal(dv, dv2)


def test_attn_bwd_random_ids(artk_lib, gpu):
    S, Hq, Hkv, D = 512, 4, 2, 128
    q, k, v = make_qkv(21, S, Hq, Hkv, D)
    g = torch.Generator().manual_seed(22)
    d_out = torch.randn(S, Hq, D, generator=g).to(torch.bfloat16)
    group = torch.randint(0, 5, (S,), generator=g)
    parent = torch.randint(0, 5, (S,), generator=g)
    _, ref_dq, ref_dk, ref_dv = attn_oracle.attention_grads(q, k, v, group, parent, d_out)
    plan = ops.attn_plan(group.to(gpu), parent.to(gpu))
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    out, lse = ops.attn_fwd(qd, kd, vd, plan)
    dq, dk, dv = ops.attn_bwd(qd, kd, vd, out, lse, d_out.to(gpu), plan)
    assert rel_l2(dq.float().cpu(), ref_dq) <= 1e-2
    assert rel_l2(dk.float().cpu(), ref_dk) <= 1e-2
    assert rel_l2(dv.float().cpu(), ref_dv) <= 1e-2


def test_packed_attention_autograd(artk_lib, gpu):
    """The module-level entry: batch of two packed rows, [B, H, S, D] storage, autograd."""
    from art_amd.attention import attention_plans, packed_attention
    B, S, Hq, Hkv, D = 2, 256, 4, 2, 64
    g = torch.Generator().manual_seed(31)
    mk = lambda H: torch.randn(B, H, S, D, generator=g).to(torch.bfloat16)
    q, k, v, d_out = mk(Hq), mk(Hkv), mk(Hkv), mk(Hq)
    ids = [synthetic.packed_row_ids(40 + b, S, 1 + b, 20, 2, 50) for b in range(B)]
    group = torch.stack([i[0] for i in ids])
    parent = torch.stack([i[1] for i in ids])
    plans = attention_plans(group.to(gpu), parent.to(gpu))
    qd, kd, vd = (t.to(gpu).requires_grad_(True) for t in (q, k, v))
    out = packed_attention(qd.transpose(1, 2), kd.transpose(1, 2), vd.transpose(1, 2), plans)
    out.backward(d_out.to(gpu).transpose(1, 2))
    for b in range(B):
        sh = lambda t: t[b].permute(1, 0, 2)
        ref_out, ref_dq, ref_dk, ref_dv = attn_oracle.attention_grads(sh(q), sh(k), sh(v), group[b], parent[b],
                                                                      sh(d_out))
        assert rel_l2(out[b].float().cpu(), ref_out) <= 1e-2
        assert rel_l2(qd.grad[b].float().cpu().permute(1, 0, 2), ref_dq) <= 1e-2
        assert rel_l2(kd.grad[b].float().cpu().permute(1, 0, 2), ref_dk) <= 1e-2
        assert rel_l2(vd.grad[b].float().cpu().permute(1, 0, 2), ref_dv) <= 1e-2


@pytest.mark.parametrize("S", [200, 300, 1000])
def test_packed_attention_any_row_length(artk_lib, gpu, S):
    """Row lengths that are not a multiple of the kernels' 256: the wrapper appends positions
    nothing real can see; out and gradients of the real positions match the oracle on the
    unpadded row (padding ids of the packer, -1, included at the end of the real row)."""
    from art_amd.attention import attention_plans, packed_attention
    print(f"packed_attention S={S}", flush=True)
    Hq, Hkv, D = 4, 2, 64
    g = torch.Generator().manual_seed(77 + S)
    mk = lambda H: torch.randn(S, H, D, generator=g).to(torch.bfloat16)
    q, k, v, d_out = mk(Hq), mk(Hkv), mk(Hkv), mk(Hq)
    group, parent = synthetic.packed_row_ids(50 + S, S, 2, S // 10, 2, S // 6)
    assert (group == -1).any()  # the packer's own padding is part of the case
    plans = attention_plans(group.to(gpu), parent.to(gpu))
    assert plans[0].S % 256 == 0 and plans[0].S - S < 256
    qd, kd, vd = (t.to(gpu).requires_grad_(True) for t in (q, k, v))
    out = packed_attention(qd, kd, vd, plans)
    assert out.shape == (S, Hq, D)
    out.backward(d_out.to(gpu))
    ref_out, ref_dq, ref_dk, ref_dv = attn_oracle.attention_grads(q, k, v, group, parent, d_out)
    assert rel_l2(out.float().cpu(), ref_out) <= 1e-2
    assert rel_l2(qd.grad.float().cpu(), ref_dq) <= 1e-2
    assert rel_l2(kd.grad.float().cpu(), ref_dk) <= 1e-2
    assert rel_l2(vd.grad.float().cpu(), ref_dv) <= 1e-2


def test_attn_full_size_windows(artk_lib, gpu):
    """Row of 16384 positions at the 7B head shape (28 query / 4 key-value heads of
    128): windows of queries against the oracle, and properties that need no
    oracle (padding rows see only padding; the first token of a completion
    attends to its prompt and itself)."""
    S, Hq, Hkv, D = 16384, 28, 4, 128
    q, k, v = make_qkv(77, S, Hq, Hkv, D)
    group, parent = synthetic.packed_row_ids(78, S, 8, 128, 4, 470)   # 8 * 2008 = 16064, rest padding
    plan = ops.attn_plan(group.to(gpu), parent.to(gpu))
    out, lse = ops.attn_fwd(q.to(gpu), k.to(gpu), v.to(gpu), plan)
    out, lse = out.float().cpu(), lse.cpu()
    for start in (0, 2008 - 30, 128 + 470 - 8, 16064 - 40, S - 64):
        rows = torch.arange(start, start + 64)
        ref_out, ref_lse = attn_oracle.attention_rows(q, k, v, group, parent, rows)
        assert (lse[:, rows] - ref_lse).abs().max().item() <= 2e-3
        assert rel_l2(out[rows], ref_out) <= 1e-2
    # the first padding position sees only itself: out = v of that position
    first_pad = 16064
    assert torch.equal(out[first_pad, :7].to(torch.bfloat16), v[first_pad, 0].expand(7, D))
    # determinism
    out2, _ = ops.attn_fwd(q.to(gpu), k.to(gpu), v.to(gpu), plan)
    assert torch.equal(out2.float().cpu(), out)


def test_attn_bwd_full_size_against_oracle(artk_lib, gpu):
    """Backward at the full 7B shape (16384 positions, 28 query / 4 key-value heads of 128): dQ, dK and
    dV of the WHOLE row against the oracle, which runs here on the GPU in fp32, 512 queries at a time
    (autograd accumulates dK and dV over the chunks), plus the two sums that need no oracle."""
    print("attention backward S=16384, 28/4 x 128", flush=True)
    S, Hq, Hkv, D = 16384, 28, 4, 128
    q, k, v = make_qkv(177, S, Hq, Hkv, D)
    g = torch.Generator().manual_seed(178)
    d_out = torch.randn(S, Hq, D, generator=g).to(torch.bfloat16)
    group, parent = synthetic.packed_row_ids(179, S, 8, 128, 4, 470)   # 8 * 2008 = 16064, rest padding
    qd, kd, vd, dod = q.to(gpu), k.to(gpu), v.to(gpu), d_out.to(gpu)
    gd, pd = group.to(gpu), parent.to(gpu)
    plan = ops.attn_plan(gd, pd)
    out, lse = ops.attn_fwd(qd, kd, vd, plan)
    dq, dk, dv = ops.attn_bwd(qd, kd, vd, out, lse, dod, plan)
    qr = qd.float().requires_grad_(True)
    kr = kd.float().requires_grad_(True)
    vr = vd.float().requires_grad_(True)
    for start in range(0, S, 512):
        rows = torch.arange(start, start + 512, device=gpu)
        ref_out, ref_lse = attn_oracle.attention_rows(qr, kr, vr, gd, pd, rows)
        assert (lse[:, rows] - ref_lse.detach()).abs().max().item() <= 2e-3
        assert rel_l2(out[rows].float(), ref_out.detach()) <= 1e-2
        ref_out.backward(dod[rows].float())
    assert rel_l2(dq.float(), qr.grad) <= 1e-2
    assert rel_l2(dk.float(), kr.grad) <= 1e-2
    assert rel_l2(dv.float(), vr.grad) <= 1e-2
    # per completion block too, so that an error confined to a few rows cannot hide in the norm
    for lo in range(0, S, 2048):
        assert rel_l2(dk[lo:lo + 2048].float(), kr.grad[lo:lo + 2048]) <= 1.5e-2
        assert rel_l2(dv[lo:lo + 2048].float(), vr.grad[lo:lo + 2048]) <= 1.5e-2
        assert rel_l2(dq[lo:lo + 2048].float(), qr.grad[lo:lo + 2048]) <= 1.5e-2
    rep = Hq // Hkv
    want_dv = d_out.double().view(S, Hkv, rep, D).sum((0, 2))            # each softmax row sums to 1
    got_dv = dv.double().cpu().sum(0)
    assert ((got_dv - want_dv).norm() / want_dv.norm()).item() <= 1e-2
    dk64 = dk.double().cpu()                                             # each row of dS sums to 0
    assert dk64.sum(0).abs().max().item() <= 2.0 ** -8 * dk64.abs().sum(0).max().item()


def test_attn_longest_row_windows_and_sums(artk_lib, gpu):
    """The longest row the kernels take (65536 positions, no padding): forward and dQ on windows
    of queries against the oracle, and two sums over the whole row that need no oracle:
    sum_j dV_j = sum over the group's heads and all queries of dO (each softmax row sums to 1)
    and sum_j dK_j = 0 (each row of dS sums to 0)."""
    print("attention S=65536", flush=True)
    S, Hq, Hkv, D = 65536, 4, 2, 64
    q, k, v = make_qkv(91, S, Hq, Hkv, D)
    g = torch.Generator().manual_seed(92)
    d_out = torch.randn(S, Hq, D, generator=g).to(torch.bfloat16)
    group, parent = synthetic.packed_row_ids(93, S, 16, 256, 4, 960)   # 16 * 4096 = 65536
    plan = ops.attn_plan(group.to(gpu), parent.to(gpu))
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    out, lse = ops.attn_fwd(qd, kd, vd, plan)
    dq, dk, dv = ops.attn_bwd(qd, kd, vd, out, lse, d_out.to(gpu), plan)
    out_c, lse_c, dq_c = out.float().cpu(), lse.cpu(), dq.float().cpu()
    for start in (0, 4096 - 32, 32768 + 256 + 960 - 8, S - 64):
        rows = torch.arange(start, start + 64)
        qw = q.float().clone().requires_grad_(True)
        ref_out, ref_lse = attn_oracle.attention_rows(qw, k, v, group, parent, rows)
        ref_out.backward(d_out[rows].float())
        assert (lse_c[:, rows] - ref_lse.detach()).abs().max().item() <= 2e-3
        assert rel_l2(out_c[rows], ref_out.detach()) <= 1e-2
        assert rel_l2(dq_c[rows], qw.grad[rows]) <= 1e-2
    rep = Hq // Hkv
    want_dv = d_out.double().view(S, Hkv, rep, D).sum((0, 2))            # [Hkv, D]
    got_dv = dv.double().cpu().sum(0)
    assert ((got_dv - want_dv).norm() / want_dv.norm()).item() <= 1e-2
    # rounding only: bf16 stores of 65536 rows, each about |dK_j| * 2^-9
    dk64 = dk.double().cpu()
    assert dk64.sum(0).abs().max().item() <= 2.0 ** -8 * dk64.abs().sum(0).max().item()


def test_attn_bwd_mixed_light_and_heavy_key_blocks(artk_lib, gpu):
    """Grouped-query backward where early key blocks are seen by many (tile, head)
    pairs (one work-group per head, fp32 partials, reduction) and late ones by few
    (one work-group for the whole group, direct store)."""
    S, Hq, Hkv, D = 1024, 8, 1, 64
    q, k, v = make_qkv(61, S, Hq, Hkv, D)
    g = torch.Generator().manual_seed(62)
    d_out = torch.randn(S, Hq, D, generator=g).to(torch.bfloat16)
    group, parent = synthetic.packed_row_ids(63, S, 1, 100, 1, 924)
    _, ref_dq, ref_dk, ref_dv = attn_oracle.attention_grads(q, k, v, group, parent, d_out)
    plan = ops.attn_plan(group.to(gpu), parent.to(gpu))
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    out, lse = ops.attn_fwd(qd, kd, vd, plan)
    # both regimes present with the threshold of large rows: first key block heavy, last one light
    assert (S // 64) * Hq > 64 and 2 * Hq <= 64
    results = {}
    for knob in (64, 0):  # the library picks 0 by itself for a row this short
        artk_lib.artk_attn_bwd_tuning(knob)
        try:
            dq, dk, dv = ops.attn_bwd(qd, kd, vd, out, lse, d_out.to(gpu), plan)
        finally:
            artk_lib.artk_attn_bwd_tuning(-1)
        assert rel_l2(dq.float().cpu(), ref_dq) <= 1e-2
        assert rel_l2(dk.float().cpu(), ref_dk) <= 1e-2
        assert rel_l2(dv.float().cpu(), ref_dv) <= 1e-2
        results[knob] = (dk, dv)
    assert rel_l2(results[64][0].float(), results[0][0].float()) <= 4e-3


@pytest.mark.parametrize("S,Hq,Hkv,D", [(1792, 7, 1, 64), (2304, 7, 1, 64), (2304, 4, 2, 128), (2304, 2, 2, 128),
                                         (2304, 16, 2, 64)])
def test_attn_dense_causal_row(artk_lib, gpu, S, Hq, Hkv, D):
    """One conversation: the lists of 28 key blocks average 14.5 query tiles (several heads per work-group of dK/dV), those
    of 36 average 18.5 (one); 18 query blocks do not divide by the XCDs that share a key/value head; with 16 heads an XCD
    has 40 work-groups, 8 of them second on their CU."""
    print("attention dense row", S, Hq, Hkv, D, flush=True)
    q, k, v = make_qkv(S + Hq, S, Hq, Hkv, D)
    d_out = torch.randn(S, Hq, D, generator=torch.Generator().manual_seed(S)).to(torch.bfloat16)
    ids = torch.zeros(S, dtype=torch.int64)
    ref = attn_oracle.attention_grads(q, k, v, ids, ids, d_out)
    plan = ops.attn_plan(ids.to(gpu), ids.to(gpu))
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    out, lse = ops.attn_fwd(qd, kd, vd, plan)
    for got, want in zip((out, *ops.attn_bwd(qd, kd, vd, out, lse, d_out.to(gpu), plan)), ref):
        assert rel_l2(got.float().cpu(), want) <= 1e-2


@pytest.mark.parametrize("B,S,Hq,Hkv,D,head_major", [
    (3, 5, 2, 1, 64, False),       # a handful of positions (one alone has a zero gradient, no relative error)
    (2, 65, 4, 4, 128, True),      # one head per group; one position in the second key tile
    (3, 257, 6, 2, 64, True),      # one position in the second padded block
    (2, 700, 7, 1, 128, False),
])
def test_packed_attention_ragged_batch(artk_lib, gpu, B, S, Hq, Hkv, D, head_major):
    """A batch of rows whose length is no multiple of a tile, in one call: nothing outside a head's S rows may
    be read (the tensors are embedded in NaN) and every row equals the oracle.  Plans made together and plans
    made one by one (a call per row) agree bit for bit."""
    from art_amd.attention import attention_plans, packed_attention
    print("ragged batch", B, S, Hq, Hkv, D, head_major, flush=True)
    g = torch.Generator().manual_seed(B * 1000 + S)
    data = [torch.randn(B, S, H, D, generator=g).to(torch.bfloat16) for H in (Hq, Hkv, Hkv, Hq)]

    def embed(t):   # the same values inside a larger tensor of NaN
        b, s, h, d = t.shape
        big = torch.full((b, h + 1, s + 9, d) if head_major else (b, s + 9, h + 1, d), float("nan"),
                         dtype=torch.bfloat16, device=gpu)
        view = big[:, :h, :s].transpose(1, 2) if head_major else big[:, :s, :h]
        view.copy_(t)
        return view

    ids = [synthetic.packed_row_ids(60 + b, S, 1, max(S // 5, 1), 2, S // 4) for b in range(B)]
    group, parent = torch.stack([i[0] for i in ids]), torch.stack([i[1] for i in ids])
    q, k, v, up = (embed(t) for t in data)
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    plans = attention_plans(group.to(gpu), parent.to(gpu))
    out = packed_attention(*leaves, plans)
    grads = torch.autograd.grad(out, leaves, up)
    single = [attention_plans(group[b].to(gpu), parent[b].to(gpu))[0] for b in range(B)]
    out1 = packed_attention(*leaves, single)
    assert torch.equal(out1, out)
    for b in range(B):
        ref = attn_oracle.attention_grads(*(t[b] for t in data[:3]), group[b], parent[b], data[3][b])
        for got, want in zip((out, *grads), ref):
            assert torch.isfinite(got[b]).all() and rel_l2(got[b].float().cpu(), want) <= 1e-2


def test_attn_batch_backward_in_several_launches(artk_lib, gpu):
    """Three rows whose partial sums of dK and dV do not fit the shared scratch together: two launches, of two rows and
    of one, and each row's gradients are those of a call of its own (to the rounding of another order of heads)."""
    from art_amd.attention import attention_plans, packed_attention
    B, S, Hq, Hkv, D = 3, 8000, 28, 4, 128
    assert 2 * 2 * 4 * 8192 * Hq * D <= 448 << 20 < 3 * 2 * 4 * 8192 * Hq * D
    print("attention batch", B, S, Hq, Hkv, D, flush=True)
    g = torch.Generator(device=gpu).manual_seed(5)
    data = [torch.randn(B, S, H, D, generator=g, device=gpu).to(torch.bfloat16) for H in (Hq, Hkv, Hkv, Hq)]
    ids = [synthetic.packed_row_ids(70 + b, S, 1 + b, 100, 2, 600) for b in range(B)]
    group, parent = (torch.stack([i[j] for i in ids]).to(gpu) for j in (0, 1))

    def grads(rows):
        leaves = [t[rows].detach().requires_grad_(True) for t in data[:3]]
        return torch.autograd.grad(packed_attention(*leaves, attention_plans(group[rows], parent[rows])), leaves,
                                   data[3][rows])

    batch = grads(slice(None))
    for b in range(B):
        for got, want in zip(batch, grads(slice(b, b + 1))):
            assert rel_l2(got[b].float(), want[0].float()) <= 4e-3


LAYOUT_VIEWS = {
    # views whose values, [2, S, H, 64], the kernels cannot address as they lie
    "every_other_d": lambda t: torch.stack([t, t], -1).flatten(-2)[..., ::2],
    "odd_stride": lambda t: torch.nn.functional.pad(t, (0, 3))[..., :-3],
    "odd_pointer": lambda t: torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape),
    "one_head_for_all": lambda t: t[:, :, :1].expand(t.shape),
}


@pytest.mark.parametrize("view", list(LAYOUT_VIEWS))
@pytest.mark.parametrize("S", [1, 300])
def test_packed_attention_any_layout(artk_lib, gpu, S, view):
    """Rows that are no multiple of 256 may have any strides and alignment, and the upstream gradient may at any
    length: the same bits as contiguous copies give.  Whole blocks with such strides are refused."""
    from art_amd.attention import attention_plans, packed_attention
    print("attention layout", S, view, flush=True)
    make = LAYOUT_VIEWS[view]
    g = torch.Generator().manual_seed(S)
    data = [torch.randn(2, S, H, 64, generator=g).to(torch.bfloat16).to(gpu) for H in (4, 2, 2, 4)]
    odd = [make(t) for t in data]
    plain = [t.clone(memory_format=torch.contiguous_format) for t in odd]
    ids = torch.zeros(2, S, dtype=torch.int64, device=gpu)
    plans = attention_plans(ids, ids)

    def run(q, k, v, up):
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
        out = packed_attention(*leaves, plans)
        return [out.detach(), *torch.autograd.grad(out, leaves, up)]

    want = run(*plain)
    for got, ref in zip(run(*odd), want):
        assert torch.equal(got, ref)
    whole = [torch.randn(2, 256, H, 64, generator=g).to(torch.bfloat16).to(gpu) for H in (4, 2, 2, 4)]
    ids = torch.zeros(2, 256, dtype=torch.int64, device=gpu)
    plans = attention_plans(ids, ids)
    for got, ref in zip(run(*whole[:3], make(whole[3])), run(*whole[:3], make(whole[3]).clone())):
        assert torch.equal(got, ref)
    with pytest.raises(ValueError):
        packed_attention(make(whole[0]), *whole[1:3], plans)


def plan_arrays(plan, S):
    """The arrays of a row's plan (S: padded) by name, from the layout the library documents by its allocator: in order,
    each at the next multiple of 256 bytes."""
    q, k = S // 128, S // 64
    buf, off, out = plan.buf.cpu(), 0, {}
    for name, n, shape in (("gc", S, (S,)), ("pc", S, (S,)), ("info", q * k, (q, k)), ("list", q * k, (q, k)), ("cnt", q, (q,)),
                           ("order", q, (q,)), ("info2", k * k, (k, k)), ("list2", k * k, (k, k)), ("cnt2", k, (k,)),
                           ("order2", k, (k,)), ("total2", 1, (1,)), ("uni", S // 16, (S // 32, 2)), ("heads", S, (S,)),
                           ("n_heads", 1, (1,))):
        off = (off + 255) // 256 * 256
        out[name] = buf[off:off + 4 * n].view(torch.int32).view(*shape)
        off += 4 * n
    return out


@pytest.mark.parametrize("S", [1, 31, 64, 130, 256, 257, 700, 1009, 1024])
@pytest.mark.parametrize("ids", ["packed", "random", "one"])
def test_plan_of_a_short_row_is_that_of_a_long_one(artk_lib, gpu, S, ids):
    """Rows of up to 1024 positions have their plan from two launches (a work-group per query block that finds the codes of
    the row for itself, then one per row that orders the tiles), longer ones from a chain of five.  Continued by positions
    whose ids occur nowhere else, a short row becomes a long one with the same visibility."""
    print(f"short plan S={S} ids={ids}", flush=True)
    g = torch.Generator().manual_seed(S)
    if ids == "packed" and S >= 130:
        group, parent = synthetic.packed_row_ids(S, S, 2, S // 20 + 1, 3, S // 8)
    elif ids == "one":
        group, parent = torch.zeros(S, dtype=torch.int64), torch.zeros(S, dtype=torch.int64)
    else:
        group, parent = (torch.randint(-4, 5, (S,), generator=g) * (1 << 40) for _ in range(2))
    pad, L = (S + 255) // 256 * 256, 2048
    more = torch.arange(L - S) + (1 << 50)
    rows = lambda a, b: ops.attn_plan_rows(torch.stack([a, a.flip(0)]).to(gpu), torch.stack([b, b.flip(0)]).to(gpu))
    short = rows(group, parent)
    long = rows(torch.cat([group, more]), torch.cat([parent, more + (1 << 51)]))
    long_flip = ops.attn_plan_rows(torch.cat([group.flip(0), more]).unsqueeze(0).to(gpu),
                                   torch.cat([parent.flip(0), more + (1 << 51)]).unsqueeze(0).to(gpu))
    for plan, ref in ((short[0], long[0]), (short[1], long_flip[0])):
        a, b = plan_arrays(plan, pad), plan_arrays(ref, L)
        assert torch.equal(a["gc"][:S], b["gc"][:S]) and torch.equal(a["pc"], b["pc"][:pad])
        for t, q in (("", pad // 128), ("2", pad // 64)):
            k = pad // 64
            assert torch.equal(a["info" + t], b["info" + t][:q, :k])
            assert torch.equal(a["cnt" + t], b["cnt" + t][:q])
            for i in range(q):
                n = int(a["cnt" + t][i])
                assert torch.equal(a["list" + t][i, :n], b["list" + t][i, :n])
            cnt = a["cnt" + t].tolist()
            assert a["order" + t].tolist() == sorted(range(q), key=lambda i: (-cnt[i], -i))
        assert int(a["total2"]) == int(a["cnt2"].sum())
        n = int(a["n_heads"])
        assert n == int((b["heads"][:int(b["n_heads"])] < S).sum()) and torch.equal(a["heads"][:n], b["heads"][:n])
        whole = S // 32
        assert torch.equal(a["uni"][:whole], b["uni"][:whole])


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S", [31, 32, 33, 64, 96, 160, 480])
def test_attn_steps_of_32_keys(artk_lib, gpu, S, D):
    """Runs of 32 positions that belong to two groups by turns, and positions of the second that see the first one's: whole
    halves of a 64-key tile are invisible to a work-group (first, last, alone in the list) or to some of its waves."""
    from art_amd.attention import attention_plans, packed_attention
    print("attention steps of 32 keys", S, D, flush=True)
    Hq, Hkv = 4, 2
    q, k, v = make_qkv(S + D, S, Hq, Hkv, D)
    d_out = torch.randn(S, Hq, D, generator=torch.Generator().manual_seed(S)).to(torch.bfloat16)
    run = torch.arange(S) // 32
    for group, parent in ((run % 2, run % 2), (run % 2, (run % 3 == 2).long()), (run % 5, (run + 3) % 5), (run, run)):
        ref_out, ref_dq, ref_dk, ref_dv = attn_oracle.attention_grads(q, k, v, group, parent, d_out)
        plans = attention_plans(group.to(gpu), parent.to(gpu))
        leaves = [t.to(gpu).requires_grad_(True) for t in (q, k, v)]
        out = packed_attention(*leaves, plans)
        got = [out.detach(), *torch.autograd.grad(out, leaves, d_out.to(gpu))]
        for a, b in zip(got, (ref_out, ref_dq, ref_dk, ref_dv)):
            assert rel_l2(a.float().cpu(), b) <= 1e-2


@pytest.mark.parametrize("S,Hq,Hkv,D,layout", [
    (2560, 16, 2, 128, (4, 60, 4, 130)),    # more work-groups of dK/dV than the GPU holds, XCDs shared by two key/value heads
    (2816, 15, 3, 128, (2, 90, 5, 250)),    # key/value heads that do not divide the XCDs
    (3328, 16, 1, 64, (3, 500, 2, 250)),    # shares of 1 to 16 heads, all XCDs on one key/value head
    (2816, 16, 16, 64, (4, 60, 4, 130)),    # nothing to share
])
def test_attn_bwd_numbers_work_groups_share_by_share(artk_lib, gpu, S, Hq, Hkv, D, layout):
    print("attention shares", S, Hq, Hkv, D, flush=True)
    q, k, v = make_qkv(S + Hq, S, Hq, Hkv, D)
    d_out = torch.randn(S, Hq, D, generator=torch.Generator().manual_seed(S)).to(torch.bfloat16)
    group, parent = synthetic.packed_row_ids(S, S, *layout)
    ref = attn_oracle.attention_grads(q, k, v, group, parent, d_out)[1:]
    plan = ops.attn_plan(group.to(gpu), parent.to(gpu))
    qd, kd, vd, up = (t.to(gpu) for t in (q, k, v, d_out))
    out, lse = ops.attn_fwd(qd, kd, vd, plan)
    for knob in (-1, 8, 64):  # (the library's own shares, and two that mix whole groups with single heads)
        artk_lib.artk_attn_bwd_tuning(knob)
        try:
            got, again = (ops.attn_bwd(qd, kd, vd, out, lse, up, plan) for _ in range(2))
        finally:
            artk_lib.artk_attn_bwd_tuning(-1)
        for a, b, c in zip(got, ref, again):
            assert rel_l2(a.float().cpu(), b) <= 1e-2
            assert torch.equal(a, c)


def out_of_rounded_p(s, v, keys, lazy):
    """[S, D] in 64 bits but for P, rounded to bf16 below a reference that waves of 32 queries move to their maximum over `keys` keys
    where one of their scores is 2^lazy above it.  s: masked scores in units of log2."""
    S, n = s.shape[0], -(-s.shape[0] // 64) * 64
    w = torch.nn.functional.pad(s, (0, n - S, 0, n - S), value=float("-inf")).view(n // 32, 32, n)
    v = torch.nn.functional.pad(v, (0, 0, 0, n - S))
    m, total, o = w.new_full((n // 32, 32), -1e30), w.new_zeros(n // 32, 32), w.new_zeros(n // 32, 32, v.shape[1])
    fresh = torch.ones(n // 32, dtype=torch.bool, device=s.device)   # the first keys that a wave sees move it at once
    for k0 in range(0, n, keys):
        x = w[:, :, k0:k0 + keys]
        top = x.amax(2)
        seen = torch.isfinite(top).any(1)
        move = (top > m + torch.where(fresh, 0.0, lazy)[:, None]).any(1) & seen
        new = torch.where(move[:, None], torch.maximum(m, top), m)
        alpha = torch.exp2(m - new)
        e = torch.exp2(x - new[..., None]).float()
        o = o * alpha[..., None] + e.to(torch.bfloat16).double() @ v[k0:k0 + keys]
        total, m, fresh = total * alpha + e.double().sum(2), new, fresh & ~seen
    return (o / total[..., None]).view(n, -1)[:S]


@pytest.mark.parametrize("std", [1.0, 2.0, 4.0, 8.0])
def test_attn_fwd_is_as_exact_as_steps_of_64_keys(artk_lib, gpu, std):
    """out at a head dimension of 128 is no farther from 64 bits than one whose P is rounded below a reference that follows the
    maximum of 64 keys from 2^8 on, be the scores flat or peaked."""
    S, Hq, Hkv, D = 2531, 28, 4, 128
    print("attention against 64 bits", std, flush=True)
    q, k, v = (t.to(gpu) for t in make_qkv(int(std), S, Hq, Hkv, D))
    q = (q.float() * std).to(torch.bfloat16)
    group, parent = (t.to(gpu) for t in synthetic.packed_row_ids(7, S, 2, 150, 4, 260))
    from art_amd.attention import attention_plans, packed_attention
    with torch.no_grad():
        out = packed_attention(q, k, v, attention_plans(group, parent))
    i = torch.arange(S, device=gpu)
    hidden = (i[None] > i[:, None]) | ((group[:, None] != group[None]) & (parent[:, None] != group[None]))
    err = torch.zeros(2, dtype=torch.float64, device=gpu)
    for h in range(Hq):
        kh, vh = (t[:, h * Hkv // Hq].double() for t in (k, v))
        s = (q[:, h].double() @ kh.t().contiguous() * D ** -0.5).masked_fill_(hidden, float("-inf"))
        ref = torch.softmax(s, 1) @ vh
        other = out_of_rounded_p(s * 1.4426950408889634, vh, 64, 8.0).to(torch.bfloat16)
        err += torch.stack([(t.double() - ref).pow(2).sum() for t in (out[:, h], other)])
    assert err[0] <= err[1], err.sqrt().tolist()


def test_attn_row_is_the_same_in_any_batch(artk_lib, gpu):
    """A row that fills the GPU only together with another: out and dQ (which reads lse) are those of the row alone, bit for bit,
    and of a call with some of its heads."""
    from art_amd.attention import attention_plans, packed_attention
    B, S, Hq, Hkv, D = 2, 2531, 16, 2, 128
    print("attention row in a batch", flush=True)
    g = torch.Generator(device=gpu).manual_seed(3)
    data = [torch.randn(B, S, H, D, generator=g, device=gpu).to(torch.bfloat16) for H in (Hq, Hkv, Hkv, Hq)]
    ids = [synthetic.packed_row_ids(80 + b, S, 2, 150, 4, 260) for b in range(B)]
    group, parent = (torch.stack([i[j] for i in ids]).to(gpu) for j in (0, 1))

    def call(rows, heads=slice(None), kv_heads=slice(None)):
        leaves = [t[rows, :, h].detach().requires_grad_(True) for t, h in zip(data, (heads, kv_heads, kv_heads))]
        out = packed_attention(*leaves, attention_plans(group[rows], parent[rows]))
        return out.detach(), torch.autograd.grad(out, leaves, data[3][rows, :, heads])[0]

    batch = call(slice(None))
    for b in range(B):
        for got, want in zip(batch, call(slice(b, b + 1))):
            assert torch.equal(got[b], want[0])
        for got, want in zip(batch, call(slice(b, b + 1), slice(0, Hq // Hkv), slice(0, 1))):
            assert torch.equal(got[b, :, :Hq // Hkv], want[0])


@pytest.mark.parametrize("D", [64, 128])
def test_attn_bwd_mask_holds_for_any_lse_and_scale(artk_lib, gpu, D):
    """P is 0 at a pair that is not visible, whatever the query's lse and the scale: dV of the keys that a poisoned query does
    not see keeps its bits, and a scale that is not positive (the forward refuses it) gives the gradients of that scale."""
    S, Hq, Hkv = 256, 4, 2
    q, k, v = make_qkv(91 + D, S, Hq, Hkv, D)
    d_out = torch.randn(S, Hq, D, generator=torch.Generator().manual_seed(5)).to(torch.bfloat16)
    ids = (torch.arange(S) >= 48).long()   # the border of the two groups lies inside a cell of 32 x 32
    plan = ops.attn_plan(ids.to(gpu), ids.to(gpu))
    print("attention backward mask", D, flush=True)

    def grads(q):
        qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
        out, lse = ops.attn_fwd(qd, kd, vd, plan)
        return ops.attn_bwd(qd, kd, vd, out, lse, d_out.to(gpu), plan)

    poisoned = q.clone()
    poisoned[60] = float("nan")
    (dq, _, dv), (dq_p, _, dv_p) = grads(q), grads(poisoned)
    assert torch.equal(dv_p[:48], dv[:48]) and torch.equal(dq_p[:48], dq[:48])
    for scale in (-0.05, 0.0):
        out, lse = attn_oracle.attention(q, k, v, ids, ids, scale)
        ref = attn_oracle.attention_grads(q, k, v, ids, ids, d_out, scale)[1:]
        got = ops.attn_bwd(*(t.to(gpu) for t in (q, k, v, out.to(torch.bfloat16), lse, d_out)), plan, scale)
        for a, b in zip(got, ref):
            assert torch.isfinite(a).all()
            if b.norm() > 0:
                assert rel_l2(a.float().cpu(), b) <= 1e-2


@pytest.mark.parametrize("head_major", [False, True])
@pytest.mark.parametrize("ids", ["dense", "scattered", "packed"])
def test_attn_fwd_steps_of_32_keys_embedded_in_nan(artk_lib, gpu, ids, head_major):
    """A row of 700 positions in more work-groups than two per CU, inside larger tensors of NaN: one causal conversation, ids
    without any order, and a packed row."""
    from art_amd.attention import attention_plans, packed_attention
    S, Hq, Hkv, D = 700, 88, 8, 128
    print("attention forward in steps of 32 keys", ids, head_major, flush=True)
    g = torch.Generator().manual_seed(S)
    data = [torch.randn(S, H, D, generator=g).to(torch.bfloat16) for H in (Hq, Hkv, Hkv, Hq)]
    group, parent = {"dense": lambda: (torch.zeros(S, dtype=torch.int64),) * 2,
                     "scattered": lambda: (torch.randint(0, 5, (S,), generator=g), torch.randint(0, 5, (S,), generator=g)),
                     "packed": lambda: synthetic.packed_row_ids(3, S, 2, 41, 3, 97)}[ids]()

    def embed(t):
        s, h, d = t.shape
        big = torch.full((h + 1, s + 9, d) if head_major else (s + 9, h + 1, d), float("nan"), dtype=torch.bfloat16, device=gpu)
        view = big[:h, :s].transpose(0, 1) if head_major else big[:s, :h]
        view.copy_(t)
        return view

    q, k, v, up = (embed(t) for t in data)
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    out = packed_attention(*leaves, attention_plans(group.to(gpu), parent.to(gpu)))
    ref = attn_oracle.attention_grads(*data[:3], group, parent, data[3])
    for got, want in zip((out.detach(), *torch.autograd.grad(out, leaves, up)), ref):
        assert torch.isfinite(got).all() and rel_l2(got.float().cpu(), want) <= 1e-2
