"""Workloads of the GRPO training path, from the smallest calls to the benchmark's own sizes.

Every case is one call (with its backward where training has one) through the package's public entry
points, on tensors that a training program has in hand at that point:

* ``grpo``      hidden states and a packed batch -> loss, metrics, logprobs and d_hidden (``fused_grpo_loss``)
* ``logprobs``  forward-only logprobs of a policy under ``no_grad`` (``_calculate_logprobs``)
* ``lora``      LoRA projections of one input, forward and backward (``LoRALinear``, ``FusedLoRALinear``)
* ``moe``       a block of experts with per-expert LoRA, forward and backward (``MoELoRAExperts``)
* ``attn``      attention over packed rows, forward and backward (``attention_plans``, ``packed_attention``)
* ``optim``     one optimizer step over all adapters (``FusedAdamW``, ``FusedAdamW8bit``)
"""
from __future__ import annotations

import math

import numpy as np
import torch

from art_amd import advantage, attention, ops, optim, quant, synthetic, train
from art_amd.lora import FusedLoRALinear, LoRALinear
from art_amd.moe import MoELoRAExperts

# (hidden size, vocabulary) of the benchmark configurations
HEADS = ((896, 151936), (2048, 151936), (3584, 152064))
# (query heads, key / value heads, head dimension) that go with them
ATTN_HEADS = ((14, 2, 64), (16, 2, 128), (28, 4, 128))


def listed():
    return [
        # one short trajectory on the 0.5B shape: the smallest training step
        {"name": "grpo_one_trajectory", "kind": "grpo", "rows": 1, "S": 317, "H": 896, "V": 151936, "traj": 1,
         "mask": 0.6, "skip": False, "beta": 0.0},
        # compute_loss' own form (only contributing positions are projected, KL term on): two odd rows, 7B shape
        {"name": "grpo_two_rows_kl", "kind": "grpo", "rows": 2, "S": 2531, "H": 3584, "V": 152064, "traj": 4,
         "mask": 0.4, "skip": True, "beta": 0.04},
        # the benchmark's default workload: 32 trajectories of 512 tokens, 7B shape, every position projected
        {"name": "grpo_full_row", "kind": "grpo", "rows": 1, "S": 16384, "H": 3584, "V": 152064, "traj": 32,
         "mask": 0.4, "skip": False, "beta": 0.0},
        # reference-policy logprobs of one packed row, 3B shape
        {"name": "logprobs_row", "kind": "logprobs", "rows": 1, "S": 4096, "H": 2048, "V": 151936},
        # q|k|v with their frozen biases over one short row, 0.5B shape: launches and latency
        {"name": "lora_qkv_short", "kind": "lora", "T": 333, "in": 896, "outs": "896,128,128", "r": 8, "bias": True,
         "base": "bf16"},
        # down projection on 4-bit base weights, 3B shape, an odd number of rows
        {"name": "lora_down_nf4", "kind": "lora", "T": 2531, "in": 11008, "outs": "2048", "r": 16, "bias": False,
         "base": "nf4"},
        # gate|up of the benchmark's LoRA workload, 3B shape
        {"name": "lora_gate_up", "kind": "lora", "T": 8192, "in": 2048, "outs": "11008,11008", "r": 8, "bias": False,
         "base": "bf16"},
        # expert block on a short row: a handful of rows per expert
        {"name": "moe_short", "kind": "moe", "T": 203, "H": 2048, "I": 768, "E": 128, "k": 8, "r": 8},
        # expert block at the benchmark's size
        {"name": "moe_full", "kind": "moe", "T": 8192, "H": 2048, "I": 768, "E": 128, "k": 8, "r": 8},
        # first layer of a step on two short rows of odd length: plans from the ids, then one layer
        {"name": "attn_two_short_rows", "kind": "attn", "rows": 2, "S": 1009, "hq": 14, "hkv": 2, "D": 64,
         "prompts": 2, "prompt": 61, "completions": 4, "completion": 107, "plan": "in the pass"},
        # one layer of the 7B shape over the benchmark's row length, plan kept from the layer before
        {"name": "attn_full_row", "kind": "attn", "rows": 1, "S": 16384, "hq": 28, "hkv": 4, "D": 128,
         "prompts": 8, "prompt": 137, "completions": 4, "completion": 461, "plan": "kept"},
        # all adapters of a 7B model, moments in 8 bits as the trainer's default optimizer keeps them
        {"name": "optim_8bit_7b", "kind": "optim", "layers": 28, "H": 3584, "I": 18944, "kv": 512, "r": 8,
         "moments": "8 bit"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("grpo", "grpo", "logprobs", "lora", "lora", "lora", "moe", "moe", "attn", "attn", "optim"))
    if kind in ("grpo", "logprobs"):
        H, V = rng.choice(HEADS)
        T = _log_int(rng, 200, 16384 if kind == "logprobs" else 13000)
        rows = rng.randint(1, 3) if T > 1000 else 1
        if kind == "logprobs":
            return {"kind": kind, "rows": rows, "S": T // rows, "H": H, "V": V}
        return {"kind": kind, "rows": rows, "S": T // rows, "H": H, "V": V,
                "traj": rng.randint(1, max(1, T // rows // 250)), "mask": round(rng.uniform(0.2, 0.7), 2),
                "skip": rng.random() < 0.5, "beta": rng.choice((0.0, 0.04))}
    if kind == "lora":
        H, I, kv = rng.choice(((896, 4864, 128), (2048, 11008, 256), (3584, 18944, 512)))
        n_in, outs = rng.choice(((H, (H, kv, kv)), (H, (I, I)), (H, (H,)), (I, (H,))))
        base = "nf4" if len(outs) == 1 and rng.random() < 0.5 else "bf16"
        T = _log_int(rng, 200, 8192)
        return {"kind": kind, "T": T, "in": n_in, "outs": ",".join(str(o) for o in outs), "r": rng.choice((8, 8, 16)),
                "bias": len(outs) == 3, "base": base}
    if kind == "moe":
        return {"kind": kind, "T": _log_int(rng, 150, 8192), "H": 2048, "I": 768, "E": rng.choice((64, 128)), "k": 8,
                "r": rng.choice((8, 16))}
    if kind == "attn":
        hq, hkv, D = rng.choice(ATTN_HEADS)
        S = _log_int(rng, 500, 16384)
        rows = 2 if S < 2000 and rng.random() < 0.5 else 1
        prompts = rng.randint(1, max(1, min(8, S // 600)))
        completions = rng.randint(2, 6)
        per = S // prompts
        prompt = rng.randint(max(8, per // 20), max(9, per // 6))
        completion = int((per - prompt) / completions * rng.uniform(0.8, 1.0))
        return {"kind": kind, "rows": rows, "S": S, "hq": hq, "hkv": hkv, "D": D, "prompts": prompts, "prompt": prompt,
                "completions": completions, "completion": completion, "plan": rng.choice(("kept", "in the pass"))}
    H, I, kv, top = rng.choice(((896, 4864, 128, 24), (2048, 11008, 256, 36), (3584, 18944, 512, 28)))
    return {"kind": kind, "layers": rng.randint(top // 4, top), "H": H, "I": I, "kv": kv,
            "r": rng.choice((8, 16)) if H < 3584 else 8, "moments": rng.choice(("8 bit", "fp32"))}


# -----------------------------------------------------------------------------
# inputs
# -----------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(gen, *shape, std=1.0, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=gen, device="cuda").mul_(std).to(dtype)


def _head_inputs(case, seed):
    """Hidden states, frozen lm_head, tokens, and the logprobs that the policy gives the next tokens (to about
    1e-2: with independent normal weights the other logits are normal with a known variance)."""
    rows, S, H, V = (case[k] for k in ("rows", "S", "H", "V"))
    gen = _gen(seed)
    lm_head = _normal(gen, V, H, std=0.02)
    tokens = torch.randint(0, V, (rows, S), generator=gen, device="cuda")
    target = torch.roll(tokens, -1, 1)
    target[:, -1] = 0
    w = lm_head[target].float()
    # a sampled token is a likely one: lean each state towards its next token's row by a random amount, so that
    # probabilities run from 1 / V to nearly 1
    lean = torch.rand(rows, S, 1, generator=gen, device="cuda") * (15.0 / (0.0004 * H))
    hidden = (torch.randn(rows, S, H, generator=gen, device="cuda") + lean * w).to(torch.bfloat16)
    z = (hidden.float() * w).sum(-1)
    rest = math.log(V) + 0.5 * 0.0004 * hidden.float().pow(2).sum(-1)
    return gen, hidden, lm_head, tokens, z - torch.logaddexp(z, rest)


def _prepare_grpo(case, seed):
    rows, S, n_traj = case["rows"], case["S"], case["traj"]
    gen, hidden, lm_head, tokens, logprob = _head_inputs(case, seed)
    host = torch.Generator().manual_seed(int(seed))
    L = S // n_traj
    mask = torch.zeros(rows, S, dtype=torch.bool)
    traj = torch.full((rows, S), -1, dtype=torch.int64)
    for row in range(rows):
        for t in range(n_traj):
            mask[row, t * L:(t + 1) * L] = synthetic.span_mask(L, int(round(case["mask"] * L)))
            traj[row, t * L:(t + 1) * L] = row * n_traj + t
    n = rows * n_traj
    rewards = torch.rand(max(n, 2), generator=host, dtype=torch.float64).numpy()
    # groups of four; a lone trajectory is one of a group whose others are in other batches
    adv = advantage.group_advantages(rewards, np.arange(len(rewards)) // 4)[:n]
    noise = lambda std: _normal(gen, rows, S, std=std, dtype=torch.float32)
    old = torch.full((rows, S), float("nan"), device="cuda")
    old[:, 1:] = (logprob + noise(0.1))[:, :-1]
    mask_d = mask.cuda()
    old = torch.where(mask_d, old, torch.full_like(old, float("nan")))
    ref = logprob + noise(0.1) if case["beta"] > 0 else None
    state = {"hidden": hidden.requires_grad_(True), "lm_head": lm_head, "tokens": tokens, "old": old,
             "adv": advantage.token_advantages(traj, adv).cuda(), "mask": mask_d,
             "weights": advantage.token_weights(mask, traj).cuda(), "ref": ref, "beta": case["beta"],
             "skip": case["skip"]}
    ops.transposed_weight(lm_head)   # the frozen weight's second layout, made once per weight
    return state


def _run_grpo(s):
    loss, metrics, logprobs = train.fused_grpo_loss(
        s["hidden"], s["lm_head"], s["tokens"], s["old"], s["adv"], s["mask"], s["weights"], ref_logprobs=s["ref"],
        beta=s["beta"], skip_inactive=s["skip"])
    (d_hidden,) = torch.autograd.grad(loss, s["hidden"])
    return {"loss": loss, "metrics": metrics, "logprobs": logprobs, "d_hidden": d_hidden}


def _prepare_logprobs(case, seed):
    _, hidden, lm_head, tokens, _ = _head_inputs(case, seed)
    return {"hidden": hidden, "lm_head_t": lm_head.t(), "ids": train.shift_tensor(tokens, 0), "chunk": case["S"]}


def _run_logprobs(s):
    with torch.no_grad():
        return train._calculate_logprobs(s["lm_head_t"], s["hidden"], s["ids"], s["chunk"])


def _prepare_lora(case, seed):
    T, n_in, r = case["T"], case["in"], case["r"]
    gen = _gen(seed)
    layers, ups = [], []
    for o in (int(v) for v in case["outs"].split(",")):
        W = _normal(gen, o, n_in, std=0.02)
        if case["base"] == "nf4":
            m = LoRALinear.from_nf4(quant.NF4Weight.from_float(W), r=r, lora_alpha=16)
        else:
            m = LoRALinear(n_in, o, r=r, lora_alpha=16, device="cuda", bias=case["bias"])
        with torch.no_grad():
            if case["base"] == "bf16":
                m.weight.copy_(W)
                ops.transposed_weight(m.weight)   # the frozen weight's second layout, made once per weight
            if case["bias"]:
                m.bias.copy_(_normal(gen, o, std=0.5))
            m.lora_A.copy_((torch.rand(r, n_in, generator=gen, device="cuda") * 2 - 1) / math.sqrt(n_in))
            m.lora_B.copy_(_normal(gen, o, r, std=0.01))
        layers.append(m)
        ups.append(_normal(gen, 1, T, o, std=0.01))
    x = _normal(gen, 1, T, n_in).requires_grad_(True)
    return {"module": FusedLoRALinear(layers) if len(layers) > 1 else layers[0], "x": x, "ups": ups,
            "params": [p for m in layers for p in (m.lora_A, m.lora_B)]}


def _run_lora(s):
    ys = s["module"](s["x"])
    ys = ys if isinstance(ys, tuple) else (ys,)
    grads = torch.autograd.grad(ys, [s["x"]] + s["params"], s["ups"])
    return {"y": list(ys), "grads": list(grads)}


def _prepare_moe(case, seed):
    T, H, I, E, k, r = (case[n] for n in ("T", "H", "I", "E", "k", "r"))
    gen = _gen(seed)
    m = MoELoRAExperts(H, I, E, k, r=r, lora_alpha=16, device="cuda")
    with torch.no_grad():
        for name, p in m.named_parameters():
            if name.endswith("weight"):
                p.copy_(torch.randn(p.shape, generator=gen, device="cuda", dtype=torch.bfloat16).mul_(0.02))
            elif name.endswith("lora_A"):
                p.copy_((torch.rand(p.shape, generator=gen, device="cuda") * 2 - 1) / math.sqrt(p.shape[2]))
            else:
                p.copy_(_normal(gen, *p.shape, std=0.01, dtype=torch.float32))
    x = _normal(gen, T, H).requires_grad_(True)
    # router logits of a trained model are uneven: some experts are liked more than others
    logits = _normal(gen, T, E, dtype=torch.float32) + _normal(gen, 1, E, std=0.5, dtype=torch.float32)
    state = {"module": m, "x": x, "logits": logits, "up": _normal(gen, T, H, std=0.01),
             "params": [p for p in m.parameters() if p.requires_grad]}
    return state


def _run_moe(s):
    y, routing = s["module"](s["x"], s["logits"])
    grads = torch.autograd.grad(y, [s["x"]] + s["params"], s["up"])
    return {"y": y, "grads": list(grads), "experts": routing.topk_idx}


def _prepare_attn(case, seed):
    rows, S, hq, hkv, D = (case[k] for k in ("rows", "S", "hq", "hkv", "D"))
    gen = _gen(seed)
    ids = [synthetic.packed_row_ids(seed + 1000 * row, S, case["prompts"], case["prompt"], case["completions"],
                                    case["completion"]) for row in range(rows)]
    group, parent = (torch.stack([i[j] for i in ids]).cuda() for j in (0, 1))
    leaf = lambda h: _normal(gen, rows, S, h, D).requires_grad_(True)
    q, k, v = leaf(hq), leaf(hkv), leaf(hkv)
    return {"q": q, "k": k, "v": v, "up": _normal(gen, rows, S, hq, D, std=0.01), "group": group, "parent": parent,
            "plans": attention.attention_plans(group, parent) if case["plan"] == "kept" else None}


def _run_attn(s):
    plans = s["plans"] if s["plans"] is not None else attention.attention_plans(s["group"], s["parent"])
    out = attention.packed_attention(s["q"], s["k"], s["v"], plans)
    grads = torch.autograd.grad(out, [s["q"], s["k"], s["v"]], s["up"])
    return {"out": out, "grads": list(grads)}


def _adapter_shapes(case):
    H, I, kv, r = (case[k] for k in ("H", "I", "kv", "r"))
    proj = {"q": (H, H), "k": (H, kv), "v": (H, kv), "o": (H, H), "gate": (H, I), "up": (H, I), "down": (I, H)}
    shapes = {}
    for layer in range(case["layers"]):
        for name, (n_in, n_out) in proj.items():
            shapes[f"{layer}.{name}.A"] = (r, n_in)
            shapes[f"{layer}.{name}.B"] = (n_out, r)
    return shapes


def _prepare_optim(case, seed):
    gen = _gen(seed)
    flat = optim.FlatParams(_adapter_shapes(case), torch.device("cuda"))
    flat.master.normal_(0.0, 0.02, generator=gen)
    flat.sync_shadow()
    opt = (optim.FusedAdamW8bit if case["moments"] == "8 bit" else optim.FusedAdamW)(flat)
    for _ in range(3):   # a run that has begun: moments are not zero
        flat.grad.normal_(0.0, 1e-3, generator=gen)
        opt.step()
    return {"flat": flat, "opt": opt}


def _run_optim(s):
    sumsq = s["opt"].step()
    flat, opt = s["flat"], s["opt"]
    moments = ([opt.state1, opt.state2, opt.absmax1, opt.absmax2] if isinstance(opt, optim.FusedAdamW8bit)
               else [opt.exp_avg, opt.exp_avg_sq])
    return {"master": flat.master, "shadow": flat.shadow, "moments": moments, "sumsq": sumsq}


_PREPARE = {"grpo": _prepare_grpo, "logprobs": _prepare_logprobs, "lora": _prepare_lora, "moe": _prepare_moe,
            "attn": _prepare_attn, "optim": _prepare_optim}
_RUN = {"grpo": _run_grpo, "logprobs": _run_logprobs, "lora": _run_lora, "moe": _run_moe, "attn": _run_attn,
        "optim": _run_optim}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    state["kind"] = case["kind"]
    return state


def run(state):
    return _RUN[state["kind"]](state)


# -----------------------------------------------------------------------------
# what a pass cannot do without, and how far another correct implementation may be off
# -----------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("grpo", "logprobs"):
        T, H, V = case["rows"] * case["S"], case["H"], case["V"]
        if kind == "logprobs":
            return {"bytes": 2 * V * H + 2 * T * H + 12 * T, "flops": 2 * T * V * H}
        active = case["mask"] * T
        projected = active if case["skip"] else T
        return {"bytes": 2 * V * H + 4 * T * H + 33 * T, "flops": 2 * (projected + active) * V * H}
    if kind == "lora":
        T, n_in, r = case["T"], case["in"], case["r"]
        n_out = sum(int(v) for v in case["outs"].split(","))
        weight = n_in * n_out * (0.5625 if case["base"] == "nf4" else 2.0)
        return {"bytes": weight + 4 * T * (n_in + n_out) + 4 * r * (n_in + n_out),
                "flops": 4 * T * n_in * n_out + 6 * T * r * (n_in + n_out)}
    if kind == "moe":
        T, H, I, E, k, r = (case[n] for n in ("T", "H", "I", "E", "k", "r"))
        used = E * (1 - (1 - k / E) ** T)
        return {"bytes": 6 * used * H * I + 8 * T * H + 4 * T * E + 24 * E * r * (H + I),
                "flops": 12 * T * k * H * I + 18 * T * k * r * (H + I)}
    if kind == "attn":
        rows, S, hq, hkv, D = (case[n] for n in ("rows", "S", "hq", "hkv", "D"))
        P, p, c, L = (case[n] for n in ("prompts", "prompt", "completions", "completion"))
        pad = S - P * (p + c * L)
        pairs = P * (p * (p + 1) // 2 + c * (L * p + L * (L + 1) // 2)) + pad * (pad + 1) // 2
        return {"bytes": rows * (8 * S * D * (hq + hkv) + 16 * S), "flops": rows * 14 * pairs * D * hq}
    n = sum(a * b for a, b in _adapter_shapes(case).values())
    return {"bytes": n * (18 if case["moments"] == "8 bit" else 30), "flops": 0}


def tolerance(case):
    """About four times what the outputs differ by from an evaluation in 64 bits on the same inputs: bf16 outputs show
    their rounding (1.7e-3 relative; 2.4e-3 for sums whose bf16 operands were rounded on the way, 4.2e-3 through the
    three products and the gating of an expert block), fp32 logprobs 2.9e-7.  The optimizer works in fp32, but a value
    next to the border of two codes (or of two bf16 values of the shadow) may fall to either side."""
    return {"grpo": {"rel": 7e-3, "max": 3e-2}, "logprobs": {"rel": 1.2e-6, "max": 5e-6},
            "lora": {"rel": 1e-2, "max": 4e-2}, "moe": {"rel": 1.7e-2, "max": 0.3}, "attn": {"rel": 1e-2, "max": 0.2},
            "optim": {"rel": 2e-5, "max": 1e-2, "differ": 5e-5}}[case["kind"]]
