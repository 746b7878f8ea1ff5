"""GPU parity of the MoE expert path: routing and permutation bit-exact, grouped
per-expert LoRA projections within rel-L2 1e-2 of the fp32 oracle."""
import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import moe_oracle  # noqa: E402

from art_amd import ops  # noqa: E402
from art_amd.moe import MoELoRAExperts  # noqa: E402

pytestmark = pytest.mark.gpu
TOL = 1e-2


def rel_l2(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


def check_routing(logits, k, gpu):
    ref = moe_oracle.route(logits, k)
    r = ops.moe_route(logits.to(gpu), k)
    assert torch.equal(r.topk_idx.cpu().long(), ref["topk_idx"])
    assert torch.equal(r.perm.cpu().long(), ref["perm"])
    assert torch.equal(r.inv_perm.cpu().long(), ref["inv_perm"])
    assert torch.equal(r.row_token.cpu().long(), ref["row_token"])
    assert torch.equal(r.offsets.cpu().long(), ref["offsets"])
    assert torch.allclose(r.topk_w.cpu(), ref["topk_w"], rtol=1e-5, atol=1e-7)
    counts = ref["offsets"][1:] - ref["offsets"][:-1]
    assert r.tile_prefix.cpu().tolist() == [0] + torch.div(counts + 255, 256, rounding_mode="floor").cumsum(0).tolist()
    assert r.blk_prefix.cpu().tolist() == [0] + torch.div(counts + 15, 16, rounding_mode="floor").cumsum(0).tolist()
    return r, ref


@pytest.mark.parametrize("T,E,k", [(64, 8, 2), (1000, 128, 8), (8192, 128, 8), (300, 5, 5), (2048, 200, 3)])
def test_route_bit_exact(artk_lib, gpu, T, E, k):
    print(f"moe route T={T} E={E} k={k}", flush=True)
    g = torch.Generator().manual_seed(T + E)
    check_routing(torch.randn(T, E, generator=g), k, gpu)


def test_route_ties_and_empty_experts(artk_lib, gpu):
    logits = torch.zeros(37, 16)          # all ties: every token picks experts 0..3
    logits[:, 9] = 1.0                    # ... except expert 9 first
    r, ref = check_routing(logits, 4, gpu)
    assert ref["topk_idx"][0].tolist() == [9, 0, 1, 2]
    assert (r.offsets.cpu()[4:9] == r.offsets.cpu()[4]).all()  # experts 3..8 empty


def test_route_nan_and_masked_logits(artk_lib, gpu):
    """Rows that are all NaN, or have fewer than k logits above -inf (masked experts, a diverged
    router), still give expert indices in [0, E): NaN counts as -inf, ties go to the lower index."""
    print("moe route with NaN / -inf rows", flush=True)
    g = torch.Generator().manual_seed(5)
    T, E, k = 517, 128, 8
    logits = torch.randn(T, E, generator=g)
    logits[3] = float("nan")
    logits[7] = float("-inf")
    logits[11, 5:] = float("-inf")               # 5 finite logits, k = 8
    logits[12, ::3] = float("nan")
    logits[13, :] = float("-inf")
    logits[13, 100] = 0.25                       # one finite logit
    logits[200:260, 64:] = float("-inf")         # half of the experts masked
    r, ref = check_routing(logits, k, gpu)
    idx = r.topk_idx.cpu()
    assert int(idx.min()) >= 0 and int(idx.max()) < E
    assert idx[3].tolist() == list(range(8)) and r.topk_w.cpu()[3].abs().max().item() == 0.0
    assert idx[13, 0].item() == 100 and r.topk_w.cpu()[13].tolist() == [1.0] + [0.0] * 7
    assert not torch.isnan(r.topk_w.cpu()).any()
    # one lane group past E (E = 200 leaves lanes of the fourth group without an expert)
    logits = torch.randn(64, 200, generator=g)
    logits[5] = float("nan")
    logits[6, 3:] = float("-inf")
    check_routing(logits, 5, gpu)


@pytest.mark.parametrize("T,E,k", [(1, 1, 1), (1, 256, 16), (63, 65, 1), (1024, 64, 1), (1025, 64, 1), (1024, 256, 4),
                                   (4097, 256, 1), (585, 130, 7)])
def test_route_edges(artk_lib, gpu, T, E, k):
    """Up to 4096 keys are sorted by one work-group, a chunk of 1024 after the other; logits of few values, so that most
    choices are ties, with signed zeros among them."""
    print(f"moe route edges T={T} E={E} k={k}", flush=True)
    g = torch.Generator().manual_seed(T + E + k)
    logits = torch.randint(-2, 3, (T, E), generator=g).float() * torch.where(torch.rand(T, E, generator=g) < 0.5, 1.0, -1.0)
    check_routing(logits, k, gpu)
    check_routing(torch.zeros(T, E), k, gpu)


def make_experts(E, n_out, n_in, r, seed):
    g = torch.Generator().manual_seed(seed)
    W = (0.02 * torch.randn(E, n_out, n_in, generator=g)).to(torch.bfloat16)
    A = ((torch.rand(E, r, n_in, generator=g) * 2 - 1) / n_in ** 0.5).to(torch.bfloat16)
    B = (0.01 * torch.randn(E, n_out, r, generator=g)).to(torch.bfloat16)
    return W, A, B


@pytest.mark.parametrize("T,H,I,E,k,use_gather", [(256, 128, 64, 8, 2, True), (300, 192, 320, 16, 4, True),
                                                  (512, 128, 256, 8, 2, False), (64, 64, 64, 32, 8, True)])
def test_grouped_lora_matches_oracle(artk_lib, gpu, T, H, I, E, k, use_gather):
    print(f"moe grouped T={T} H={H} I={I} E={E} k={k} gather={use_gather}", flush=True)
    g = torch.Generator().manual_seed(T + I)
    logits = torch.randn(T, E, generator=g)
    r, ref = check_routing(logits, k, gpu)
    n_rows = T * k
    x = torch.randn(T if use_gather else n_rows, H, generator=g).to(torch.bfloat16)
    W, A, B = make_experts(E, I, H, 8, 3)
    up = torch.randn(n_rows, I, generator=g).to(torch.bfloat16)
    y0, dx0, dA0, dB0 = moe_oracle.grouped_lora_grads(
        x, ref["row_token"] if use_gather else None, W, A, B, 2.0, ref["offsets"], up)
    gather = r.row_token if use_gather else None
    y, xa = ops.moe_lora_grouped_fwd(x.to(gpu), gather, W.to(gpu), A.to(gpu), B.to(gpu), 2.0, r)
    dx, dA, dB = ops.moe_lora_grouped_bwd(up.to(gpu), x.to(gpu), gather, ops.transpose_batched(W.to(gpu)),
                                          A.to(gpu), B.to(gpu), xa, 2.0, r)
    assert rel_l2(y.cpu().float(), y0) <= TOL
    if use_gather:  # oracle dx is per token; sum the kernel's per-row dx over each token's k rows
        dx = dx[r.inv_perm.long()].view(T, k, H).float().sum(1)
    assert rel_l2(dx.cpu().float(), dx0) <= TOL
    assert rel_l2(dA.cpu(), dA0) <= TOL
    assert rel_l2(dB.cpu(), dB0) <= TOL


@pytest.mark.parametrize("r,use_gather", [(40, True), (64, False), (16, True)])
def test_grouped_lora_ranks(artk_lib, gpu, r, use_gather):
    """Ranks other than 8: above 32 the one-pass backward runs its two-tile-per-rank shape (256-column
    chunks, two stages), with and without the row gather."""
    print(f"moe grouped rank {r} gather={use_gather}", flush=True)
    T, H, I, E, k = 384, 320, 192, 8, 2
    g = torch.Generator().manual_seed(100 + r)
    logits = torch.randn(T, E, generator=g)
    rt, ref = check_routing(logits, k, gpu)
    n_rows = T * k
    x = torch.randn(T if use_gather else n_rows, H, generator=g).to(torch.bfloat16)
    W, A, B = make_experts(E, I, H, r, 11)
    up = torch.randn(n_rows, I, generator=g).to(torch.bfloat16)
    y0, dx0, dA0, dB0 = moe_oracle.grouped_lora_grads(
        x, ref["row_token"] if use_gather else None, W, A, B, 0.5, ref["offsets"], up)
    gather = rt.row_token if use_gather else None
    y, xa = ops.moe_lora_grouped_fwd(x.to(gpu), gather, W.to(gpu), A.to(gpu), B.to(gpu), 0.5, rt)
    dx, dA, dB = ops.moe_lora_grouped_bwd(up.to(gpu), x.to(gpu), gather, ops.transpose_batched(W.to(gpu)),
                                          A.to(gpu), B.to(gpu), xa, 0.5, rt)
    assert rel_l2(y.cpu().float(), y0) <= TOL
    if use_gather:
        dx = dx[rt.inv_perm.long()].view(T, k, H).float().sum(1)
    assert rel_l2(dx.cpu().float(), dx0) <= TOL
    assert rel_l2(dA.cpu(), dA0) <= TOL
    assert rel_l2(dB.cpu(), dB0) <= TOL


@pytest.mark.parametrize("rows,H,I,r,use_gather", [
    ([0, 1, 31, 32, 33, 64, 65, 0], 64, 64, 8, True),            # one K step, half a tile of weight rows
    ([96, 97, 128, 5, 0, 17, 63, 2, 40], 192, 320, 24, False),   # fewer K steps than ring stages, a ragged weight tile
    ([129, 0, 260, 3, 0, 0, 0, 0, 0, 77], 128, 448, 8, True),    # experts in two and three passes
    ([3] * 255 + [200], 128, 128, 16, True),                     # the most experts
    ([400, 90, 90] + [0, 1, 7] * 20, 1088, 64, 8, True),         # shares of full experts, nine weight tiles over eight XCDs
    ([40], 192, 1152, 8, False),                                 # one expert
    ([300, 1, 130], 128, 192, 8, True),                          # more than 128 rows per expert: 256 x 256 tiles
    ([257, 384], 192, 320, 40, False),
])
def test_grouped_lora_rows_per_expert(artk_lib, gpu, rows, H, I, r, use_gather):
    """Row counts around the column tiles of both grouped products (32, 64, 96, 128 columns of a streaming pass, 256 of
    a tile) with K ranges shorter and longer than their rings.  TOL as above."""
    print(f"moe grouped rows {rows[:10]} H={H} I={I} r={r} gather={use_gather}", flush=True)
    E, T = len(rows), sum(rows)
    g = torch.Generator().manual_seed(T + H)
    owner = torch.repeat_interleave(torch.arange(E), torch.tensor(rows))[torch.randperm(T, generator=g)]
    logits = torch.zeros(T, E)
    logits[torch.arange(T), owner] = 1.0
    rt, ref = check_routing(logits, 1, gpu)
    off = ref["offsets"]
    assert [int(off[e + 1] - off[e]) for e in range(E)] == rows
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    W, A, B = make_experts(E, I, H, r, 21)
    up = torch.randn(T, I, generator=g).to(torch.bfloat16)
    y0, dx0, dA0, dB0 = moe_oracle.grouped_lora_grads(
        x, ref["row_token"] if use_gather else None, W, A, B, 0.5, off, up)
    gather = rt.row_token if use_gather else None
    y, xa = ops.moe_lora_grouped_fwd(x.to(gpu), gather, W.to(gpu), A.to(gpu), B.to(gpu), 0.5, rt)
    dx, dA, dB = ops.moe_lora_grouped_bwd(up.to(gpu), x.to(gpu), gather, ops.transpose_batched(W.to(gpu)),
                                          A.to(gpu), B.to(gpu), xa, 0.5, rt)
    if use_gather:
        dx = dx[rt.inv_perm.long()]
    for a, b in ((y, y0), (dx, dx0)):
        assert rel_l2(a.cpu().float(), b) <= TOL
    for e in range(E):  # no expert's rows are lost among the others'
        if rows[e]:
            assert rel_l2(y[off[e]:off[e + 1]].cpu().float(), y0[off[e]:off[e + 1]]) <= TOL
    assert rel_l2(dA.cpu(), dA0) <= TOL and rel_l2(dB.cpu(), dB0) <= TOL


def test_one_full_expert_among_many_takes_no_longer_than_alone(artk_lib, gpu):
    """All tokens on one of 128 experts: its units are spread over the GPU (on one XCD the block took four times as long
    as the same rows through a block of one expert; the streaming kernel may cost some of what the tiles of many rows
    take)."""
    T, H, I = 4000, 2048, 768
    x = torch.randn(T, H, device=gpu).to(torch.bfloat16)
    blocks = []
    for E in (1, 128):
        m = MoELoRAExperts(H, I, E, 1, r=8, lora_alpha=16, device=gpu)
        logits = torch.zeros(T, E, device=gpu)
        logits[:, 0] = 30.0
        blocks.append((m, logits))

    def median_us(m, logits):
        times = []
        for _ in range(15):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            with torch.no_grad():
                m(x, logits)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 1e3)
        return sorted(times)[7]

    alone, among = (median_us(*b) for b in blocks)
    print(f"moe one expert: alone {alone:.0f} us, among 128 {among:.0f} us", flush=True)
    assert among <= 2 * alone


@pytest.mark.parametrize("use_gather", [True, False])
def test_grouped_lora_with_empty_experts(artk_lib, gpu, use_gather):
    """Experts that no token chose: their dA_e and dB_e are exactly zero, the others match the oracle
    (the one-pass backward gives every expert its own slab of rows, here some of them empty, one of
    them longer than a 128-row tile and the first and last expert among the empty ones)."""
    print(f"moe grouped, empty experts, gather={use_gather}", flush=True)
    T, H, I, E, k = 320, 128, 192, 16, 2
    g = torch.Generator().manual_seed(5)
    logits = torch.randn(T, E, generator=g)
    dead = [0, 3, 4, 5, 15]
    logits[:, dead] = float("-inf")
    logits[:200, 7] += 8.0                      # expert 7 gets at least 200 rows
    r, ref = check_routing(logits, k, gpu)
    off = ref["offsets"]
    assert all(off[e + 1] == off[e] for e in dead) and off[8] - off[7] >= 200
    n_rows = T * k
    x = torch.randn(T if use_gather else n_rows, H, generator=g).to(torch.bfloat16)
    W, A, B = make_experts(E, I, H, 8, 9)
    up = torch.randn(n_rows, I, generator=g).to(torch.bfloat16)
    y0, dx0, dA0, dB0 = moe_oracle.grouped_lora_grads(
        x, ref["row_token"] if use_gather else None, W, A, B, 2.0, off, up)
    gather = r.row_token if use_gather else None
    y, xa = ops.moe_lora_grouped_fwd(x.to(gpu), gather, W.to(gpu), A.to(gpu), B.to(gpu), 2.0, r)
    dx, dA, dB = ops.moe_lora_grouped_bwd(up.to(gpu), x.to(gpu), gather, ops.transpose_batched(W.to(gpu)),
                                          A.to(gpu), B.to(gpu), xa, 2.0, r)
    assert rel_l2(y.cpu().float(), y0) <= TOL
    if use_gather:
        dx = dx[r.inv_perm.long()].view(T, k, H).float().sum(1)
    assert rel_l2(dx.cpu().float(), dx0) <= TOL
    assert rel_l2(dA.cpu(), dA0) <= TOL and rel_l2(dB.cpu(), dB0) <= TOL
    for e in dead:
        assert dA[e].abs().max().item() == 0.0 and dB[e].abs().max().item() == 0.0
    for e in (7, 8):
        assert rel_l2(dA[e].cpu(), dA0[e]) <= TOL and rel_l2(dB[e].cpu(), dB0[e]) <= TOL


def test_config5_gate_projection_full_size(artk_lib, gpu):
    """Benchmark config 5: 8192 tokens, hidden 2048, 128 experts, top-8, gate [768,2048]."""
    print("moe config5 gate projection", flush=True)
    T, H, I, E, k = 8192, 2048, 768, 128, 8
    g = torch.Generator().manual_seed(1005)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    logits = torch.randn(T, E, generator=g)
    r, ref = check_routing(logits, k, gpu)
    W, A, B = make_experts(E, I, H, 8, 1005)
    up = torch.randn(T * k, I, generator=g).to(torch.bfloat16)
    y0, dx0, dA0, dB0 = moe_oracle.grouped_lora_grads(x, ref["row_token"], W, A, B, 2.0, ref["offsets"], up)
    y, xa = ops.moe_lora_grouped_fwd(x.to(gpu), r.row_token, W.to(gpu), A.to(gpu), B.to(gpu), 2.0, r)
    dx, dA, dB = ops.moe_lora_grouped_bwd(up.to(gpu), x.to(gpu), r.row_token, ops.transpose_batched(W.to(gpu)),
                                          A.to(gpu), B.to(gpu), xa, 2.0, r)
    dx = dx[r.inv_perm.long()].view(T, k, H).float().sum(1)
    assert rel_l2(y.cpu().float(), y0) <= TOL
    assert rel_l2(dx.cpu(), dx0) <= TOL
    assert rel_l2(dA.cpu(), dA0) <= TOL
    assert rel_l2(dB.cpu(), dB0) <= TOL


def test_config5_down_projection_full_size(artk_lib, gpu):
    """Benchmark config 5, down projection [2048,768] at full size: 65536 sorted rows of width 768
    (no gather: the rows are the gated activations, already in expert order), forward and backward."""
    print("moe config5 down projection", flush=True)
    T, H, I, E, k = 8192, 2048, 768, 128, 8
    g = torch.Generator().manual_seed(1005)
    logits = torch.randn(T, E, generator=g)
    r, ref = check_routing(logits, k, gpu)
    h = torch.randn(T * k, I, generator=g).to(torch.bfloat16)
    W, A, B = make_experts(E, H, I, 8, 2005)
    up = torch.randn(T * k, H, generator=g).to(torch.bfloat16)
    y0, dx0, dA0, dB0 = moe_oracle.grouped_lora_grads(h, None, W, A, B, 2.0, ref["offsets"], up)
    y, xa = ops.moe_lora_grouped_fwd(h.to(gpu), None, W.to(gpu), A.to(gpu), B.to(gpu), 2.0, r)
    dx, dA, dB = ops.moe_lora_grouped_bwd(up.to(gpu), h.to(gpu), None, ops.transpose_batched(W.to(gpu)),
                                          A.to(gpu), B.to(gpu), xa, 2.0, r)
    assert rel_l2(y.cpu().float(), y0) <= TOL
    assert rel_l2(dx.cpu().float(), dx0) <= TOL
    assert rel_l2(dA.cpu(), dA0) <= TOL
    assert rel_l2(dB.cpu(), dB0) <= TOL
    # per expert as well: a wrong expert boundary would hide in the global norm
    off = ref["offsets"].tolist()
    for e in (0, 1, 63, 127):
        sl = slice(off[e], off[e + 1])
        assert rel_l2(y[sl].cpu().float(), y0[sl]) <= TOL
        assert rel_l2(dx[sl].cpu().float(), dx0[sl]) <= TOL
        assert rel_l2(dA[e].cpu(), dA0[e]) <= TOL and rel_l2(dB[e].cpu(), dB0[e]) <= TOL


def test_config5_fused_gate_up_full_size(artk_lib, gpu):
    """Benchmark config 5 the way art_amd.moe.MoELoRAExperts runs gate and up: ONE grouped product
    [128, 1536, 2048] over the gathered token rows, adapters stacked to rank 16 with a block-diagonal
    B per expert.  y, dx (summed per token), dA and dB against the oracle, also expert by expert;
    gate and up halves against the oracle of each projection alone."""
    print("moe config5 fused gate|up", flush=True)
    T, H, I, E, k, r = 8192, 2048, 768, 128, 8, 8
    g = torch.Generator().manual_seed(1005)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    logits = torch.randn(T, E, generator=g)
    rt, ref = check_routing(logits, k, gpu)
    Wg, Ag, Bg = make_experts(E, I, H, r, 1005)
    Wu, Au, Bu = make_experts(E, I, H, r, 3005)
    W = torch.cat([Wg, Wu], 1).contiguous()
    A = torch.cat([Ag, Au], 1).contiguous()
    B = torch.zeros(E, 2 * I, 2 * r, dtype=torch.bfloat16)
    B[:, :I, :r], B[:, I:, r:] = Bg, Bu
    up = torch.randn(T * k, 2 * I, generator=g).to(torch.bfloat16)
    y0, dx0, dA0, dB0 = moe_oracle.grouped_lora_grads(x, ref["row_token"], W, A, B, 2.0, ref["offsets"], up)
    y, xa = ops.moe_lora_grouped_fwd(x.to(gpu), rt.row_token, W.to(gpu), A.to(gpu), B.to(gpu), 2.0, rt)
    dx, dA, dB = ops.moe_lora_grouped_bwd(up.to(gpu), x.to(gpu), rt.row_token, ops.transpose_batched(W.to(gpu)),
                                          A.to(gpu), B.to(gpu), xa, 2.0, rt)
    dx = dx[rt.inv_perm.long()].view(T, k, H).float().sum(1)
    assert rel_l2(y.cpu().float(), y0) <= TOL
    assert rel_l2(dx.cpu(), dx0) <= TOL
    assert rel_l2(dA.cpu(), dA0) <= TOL
    assert rel_l2(dB.cpu(), dB0) <= TOL
    off = ref["offsets"].tolist()
    for e in (0, 1, 63, 127):
        sl = slice(off[e], off[e + 1])
        assert rel_l2(y[sl].cpu().float(), y0[sl]) <= TOL
        assert rel_l2(dA[e].cpu(), dA0[e]) <= TOL and rel_l2(dB[e].cpu(), dB0[e]) <= TOL
    # the halves are the two projections: forward and adapter gradients of gate alone
    yg0, _, dAg0, dBg0 = moe_oracle.grouped_lora_grads(x, ref["row_token"], Wg, Ag, Bg, 2.0, ref["offsets"],
                                                        up[:, :I].contiguous())
    assert rel_l2(y[:, :I].cpu().float(), yg0) <= TOL
    assert rel_l2(dA[:, :r].cpu(), dAg0) <= TOL
    assert rel_l2(dB[:, :I, :r].cpu(), dBg0) <= TOL


def test_moe_block_autograd(artk_lib, gpu):
    """The whole block (gate, up, SiLU gating, down, recombination) against torch fp32."""
    torch.manual_seed(0)
    T, H, I, E, k = 192, 128, 64, 8, 2
    mod = MoELoRAExperts(H, I, E, k, device=gpu)
    with torch.no_grad():
        for n in ("gate", "up", "down"):
            getattr(mod, f"{n}_lora_B").normal_(std=0.02)
    x = torch.randn(T, H, device=gpu).to(torch.bfloat16).requires_grad_(True)
    logits = torch.randn(T, E, device=gpu)
    y, routing = mod(x, logits)
    up = torch.randn_like(y)
    y.backward(up)
    # reference: dense per-token evaluation in fp32 on the CPU
    ref = moe_oracle.route(logits.cpu(), k)
    xr = x.detach().cpu().float().requires_grad_(True)
    P = {n: p.detach().cpu().float().requires_grad_(p.requires_grad) for n, p in mod.named_parameters()}
    assert "gate_weight" not in P and "up_weight" not in P    # one stored weight; gate / up are views of it
    assert mod.gate_weight.data_ptr() == mod.gate_up_weight.data_ptr()
    P["gate_weight"], P["up_weight"] = P["gate_up_weight"][:, :I], P["gate_up_weight"][:, I:]
    rows = xr[ref["row_token"]]
    off = ref["offsets"]
    s = mod.scaling
    gate = moe_oracle.grouped_lora(rows, P["gate_weight"], P["gate_lora_A"], P["gate_lora_B"], s, off)
    upp = moe_oracle.grouped_lora(rows, P["up_weight"], P["up_lora_A"], P["up_lora_B"], s, off)
    h = torch.nn.functional.silu(gate) * upp
    down = moe_oracle.grouped_lora(h, P["down_weight"], P["down_lora_A"], P["down_lora_B"], s, off)
    y0 = (down[ref["inv_perm"]].view(T, k, H) * ref["topk_w"].unsqueeze(-1)).sum(1)
    y0.backward(up.cpu().float())
    assert rel_l2(y.detach().cpu().float(), y0.detach()) <= 2e-2
    assert rel_l2(x.grad.cpu().float(), xr.grad) <= 2e-2
    for n in ("gate_lora_A", "gate_lora_B", "up_lora_A", "up_lora_B", "down_lora_A", "down_lora_B"):
        assert rel_l2(getattr(mod, n).grad.cpu(), P[n].grad) <= 2e-2, n


@pytest.mark.parametrize("T,H,I,E,k,r,dtype", [
    (1, 64, 64, 4, 1, 8, torch.float32),        # one row: every other expert empty
    (37, 192, 320, 5, 3, 24, torch.float32),    # nothing divides a tile; odd k
    (300, 128, 64, 3, 3, 32, torch.bfloat16),   # every expert gets every token; bf16 adapters, largest rank
    (70, 128, 128, 24, 12, 8, torch.float32),   # more slots than one round of the recombination
])
def test_moe_experts_entry_points(artk_lib, gpu, T, H, I, E, k, r, dtype):
    """artk_moe_experts_fwd / _bwd against the fp32 oracle on the same bf16-valued inputs.  2e-2 as in
    test_moe_block_autograd: three bf16-rounded products (4e-3 relative each way) in a row."""
    print("moe experts", T, H, I, E, k, r, dtype, flush=True)
    g = torch.Generator().manual_seed(T + H)
    rnd = lambda *s, std=1.0: (std * torch.randn(*s, generator=g)).to(torch.bfloat16)
    x, up, logits = rnd(T, H), rnd(T, H), torch.randn(T, E, generator=g)
    Wgu, Wd = rnd(E, 2 * I, H, std=H ** -0.5), rnd(E, H, I, std=I ** -0.5)
    P = {"gate_A": rnd(E, r, H, std=H ** -0.5), "gate_B": rnd(E, I, r, std=0.1), "up_A": rnd(E, r, H, std=H ** -0.5),
         "up_B": rnd(E, I, r, std=0.1), "down_A": rnd(E, r, I, std=I ** -0.5), "down_B": rnd(E, H, r, std=0.1)}
    ref = moe_oracle.route(logits, k)
    xr = x.float().requires_grad_(True)
    Pr = {n: p.float().requires_grad_(True) for n, p in P.items()}
    off, rows = ref["offsets"], xr[ref["row_token"]]
    gate = moe_oracle.grouped_lora(rows, Wgu[:, :I].float(), Pr["gate_A"], Pr["gate_B"], 0.5, off)
    u = moe_oracle.grouped_lora(rows, Wgu[:, I:].float(), Pr["up_A"], Pr["up_B"], 0.5, off)
    down = moe_oracle.grouped_lora(torch.nn.functional.silu(gate) * u, Wd.float(), Pr["down_A"], Pr["down_B"], 0.5, off)
    y0 = (down[ref["inv_perm"]].view(T, k, H) * ref["topk_w"].unsqueeze(-1)).sum(1)
    y0.backward(up.float())
    ad = {n: p.to(dtype).to(gpu) for n, p in P.items()}
    y, rt, saved = ops.moe_experts_fwd(x.to(gpu), logits.to(gpu), k, Wgu.to(gpu), Wd.to(gpu), ad, 0.5)
    dx, grads = ops.moe_experts_bwd(up.to(gpu), x.to(gpu), rt, saved, ops.transpose_batched(Wgu.to(gpu)),
                                    ops.transpose_batched(Wd.to(gpu)), r, 0.5)
    assert torch.equal(rt.topk_idx.cpu().long(), ref["topk_idx"].long())
    assert rel_l2(y.cpu().float(), y0.detach()) <= 2e-2
    assert rel_l2(dx.cpu().float(), xr.grad) <= 2e-2
    for n in P:
        assert grads[n].shape == P[n].shape and rel_l2(grads[n].cpu(), Pr[n].grad) <= 2e-2, n


def test_moe_parameters_changed_between_forward_and_backward(artk_lib, gpu):
    """fp32 adapters may change between forward and backward (the gradients are those of the values that the
    forward used), as long as the inputs stay."""
    from art_amd.moe import MoELoRAExperts

    torch.manual_seed(11)
    m = MoELoRAExperts(64, 64, 4, 2, r=8, lora_alpha=16, device=gpu)
    params = [p for p in m.parameters() if p.requires_grad]
    with torch.no_grad():
        for p in params:
            p.normal_(std=0.05)
    x, logits = torch.randn(9, 64, device=gpu, dtype=torch.bfloat16), torch.randn(9, 4, device=gpu)
    up = torch.randn(9, 64, device=gpu, dtype=torch.bfloat16)
    want = torch.autograd.grad(m(x, logits)[0], params, up)
    y, _ = m(x, logits)
    with torch.no_grad():
        for p in params:
            p.add_(1.0)
    for got, ref in zip(torch.autograd.grad(y, params, up), want):
        assert torch.equal(got, ref)


@pytest.mark.parametrize("E,hot", [(3, 700), (24, 4000)])
def test_moe_experts_uneven_load(artk_lib, gpu, E, hot):
    """More than a row tile per expert on average, so the skinny passes go by falling expert size: one expert with
    most of the rows, one without any, the rest of equal or nearly equal size.  Gradients against the fp32 oracle,
    2e-2 as in test_moe_experts_entry_points."""
    T, H, I, k, r = hot, 128, 64, 2, 8
    print("moe uneven", E, hot, flush=True)
    g = torch.Generator().manual_seed(E)
    rnd = lambda *s, std=1.0: (std * torch.randn(*s, generator=g)).to(torch.bfloat16)
    x, up, logits = rnd(T, H), rnd(T, H), torch.randn(T, E, generator=g)
    logits[:, 1] += 8.0
    logits[:, 0] -= 50.0
    Wgu, Wd = rnd(E, 2 * I, H, std=H ** -0.5), rnd(E, H, I, std=I ** -0.5)
    P = {"gate_A": rnd(E, r, H, std=H ** -0.5), "gate_B": rnd(E, I, r, std=0.1), "up_A": rnd(E, r, H, std=H ** -0.5),
         "up_B": rnd(E, I, r, std=0.1), "down_A": rnd(E, r, I, std=I ** -0.5), "down_B": rnd(E, H, r, std=0.1)}
    ref = moe_oracle.route(logits, k)
    off = ref["offsets"]
    assert T * k > E * 128 and int(off[1]) == 0 and int(off[2]) == T
    Pr = {n: p.float().requires_grad_(True) for n, p in P.items()}
    rows = x.float()[ref["row_token"]]
    gate = moe_oracle.grouped_lora(rows, Wgu[:, :I].float(), Pr["gate_A"], Pr["gate_B"], 0.5, off)
    u = moe_oracle.grouped_lora(rows, Wgu[:, I:].float(), Pr["up_A"], Pr["up_B"], 0.5, off)
    down = moe_oracle.grouped_lora(torch.nn.functional.silu(gate) * u, Wd.float(), Pr["down_A"], Pr["down_B"], 0.5, off)
    y0 = (down[ref["inv_perm"]].view(T, k, H) * ref["topk_w"].unsqueeze(-1)).sum(1)
    y0.backward(up.float())
    ad = {n: p.to(gpu) for n, p in P.items()}
    y, rt, saved = ops.moe_experts_fwd(x.to(gpu), logits.to(gpu), k, Wgu.to(gpu), Wd.to(gpu), ad, 0.5)
    _, grads = ops.moe_experts_bwd(up.to(gpu), x.to(gpu), rt, saved, ops.transpose_batched(Wgu.to(gpu)),
                                   ops.transpose_batched(Wd.to(gpu)), r, 0.5)
    assert rel_l2(y.cpu().float(), y0.detach()) <= 2e-2
    for n in P:
        assert rel_l2(grads[n].cpu(), Pr[n].grad) <= 2e-2, n
        assert not grads[n][0].any()   # the expert without rows


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_moe_block_takes_views_of_flat_buffers(artk_lib, gpu, dtype):
    """Adapters that are views into one buffer, and an upstream gradient that is one, at any alignment: the bits of
    the aligned call."""
    torch.manual_seed(12)
    mod = MoELoRAExperts(64, 64, 4, 2, r=8, lora_alpha=16, device=gpu)
    params = [p for p in mod.parameters() if p.requires_grad]
    with torch.no_grad():
        for p in params:
            p.data = p.normal_(std=0.05).to(dtype)
    x = torch.randn(9, 64, device=gpu, dtype=torch.bfloat16, requires_grad=True)
    logits, up = torch.randn(9, 4, device=gpu), torch.randn(9, 64, device=gpu, dtype=torch.bfloat16)

    def odd(t):
        return torch.cat([t.new_zeros(1), t.detach().flatten()])[1:].view(t.shape)

    def step(up):
        y, _ = mod(x, logits)
        return [y.detach(), *torch.autograd.grad(y, [x] + params, up)]

    want = step(up)
    for p in params:
        p.data = odd(p)
    assert all(p.data_ptr() % 16 for p in params) and odd(up).data_ptr() % 16
    for got, ref in zip(step(odd(up)), want):
        assert torch.equal(got, ref)


def test_moe_block_hooks_see_no_frozen_weights(artk_lib, gpu):
    """Hooks that move saved tensors to the host (torch.autograd.graph.save_on_cpu) see the expert block's activations, not
    its weights or their transposed copies; the gradients are the same bits.  On a stream that is not the default one."""
    torch.manual_seed(14)
    mod = MoELoRAExperts(128, 64, 4, 2, r=8, lora_alpha=16, device=gpu)
    params = [p for p in mod.parameters() if p.requires_grad]
    x = torch.randn(9, 128, device=gpu, dtype=torch.bfloat16, requires_grad=True)
    logits, up = torch.randn(9, 4, device=gpu), torch.randn(9, 128, device=gpu, dtype=torch.bfloat16)

    def step():
        y, _ = mod(x, logits)
        return [y.detach(), *torch.autograd.grad(y, [x] + params, up)]

    want = step()
    seen = []

    def pack(t):
        seen.append(tuple(t.shape))
        return t.cpu()

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(gpu)):
        got = step()
    side.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert (9, 128) in seen and not any(len(s) == 3 for s in seen)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_moe_block_without_a_backward(artk_lib, gpu, dtype):
    """Under no_grad, and where nothing needs a gradient, the block gives the same bits and makes no transposed adapters: its
    peak of memory is lower by at least their size (all else is allocated either way)."""
    E, H, I, r, T = 16, 512, 256, 16, 24
    torch.manual_seed(15)
    mod = MoELoRAExperts(H, I, E, 2, r=r, lora_alpha=16, device=gpu)
    params = [p for p in mod.parameters() if p.requires_grad]
    with torch.no_grad():
        for p in params:
            p.data = p.normal_(std=0.05).to(dtype)
    x, logits = torch.randn(T, H, device=gpu, dtype=torch.bfloat16), torch.randn(T, E, device=gpu)
    print("moe block without a backward", dtype, flush=True)

    def peak():
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        y, routing = mod(x, logits)
        torch.cuda.synchronize()
        assert y.requires_grad == (torch.is_grad_enabled() and params[0].requires_grad)
        return torch.cuda.max_memory_allocated() - before, y.detach(), routing.topk_idx

    peak()   # (the transposed frozen weights are made once)
    with_grad, want, experts = peak()
    transposed = 2 * E * (2 * r * 2 * I + H * 2 * r + r * H + I * r)
    with torch.no_grad():
        without, got, idx = peak()
    assert torch.equal(got, want) and torch.equal(idx, experts) and without <= with_grad - transposed
    for p in params:
        p.requires_grad_(False)
    assert peak()[0] == without
