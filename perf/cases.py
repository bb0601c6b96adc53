"""What this framework is timed on: the work of its users, through its public entry points.

Training steps (full, packed documents, LoRA) of Llama-type models, attention and
mixture-of-experts layers forward and backward, and prompts plus decoding through
``DecodeSession``. Models have a few layers of the real width: every layer does the
same work, and the head keeps about the share that it has in the whole model.
"""

from __future__ import annotations

import math

import torch

DEV = "cuda"
BF = torch.bfloat16
VOCAB = 32768


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def _train(name=None, *, batch, seq, hidden, inter, layers, heads, kv_heads, head_dim=128,
           vocab=VOCAB, fused=False, packed=0, rank=0):
    c = dict(kind="train", batch=batch, seq=seq, hidden=hidden, inter=inter, layers=layers,
             heads=heads, kv_heads=kv_heads, head_dim=head_dim, vocab=vocab, fused=fused,
             packed=packed, rank=rank)
    return dict(c, name=name) if name else c


def _attn(name=None, *, batch, seq, heads, kv_heads, dqk, dv):
    c = dict(kind="attn", batch=batch, seq=seq, heads=heads, kv_heads=kv_heads, dqk=dqk, dv=dv)
    return dict(c, name=name) if name else c


def _moe(name=None, *, batch, seq, hidden, inter, experts, active, shared=0, sigmoid=False):
    c = dict(kind="moe", batch=batch, seq=seq, hidden=hidden, inter=inter, experts=experts,
             active=active, shared=shared, sigmoid=sigmoid)
    return dict(c, name=name) if name else c


def _gen(name=None, *, model, batch, prompt, ragged, new, hidden, inter, layers, heads, kv_heads=0):
    c = dict(kind="gen", model=model, batch=batch, prompt=prompt, ragged=ragged, new=new,
             hidden=hidden, inter=inter, layers=layers, heads=heads, kv_heads=kv_heads)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a debug or unit-test sized step: nothing but launches and host work
        _train("train_tiny", batch=2, seq=128, hidden=256, inter=512, layers=2, heads=2,
               kv_heads=2, vocab=1024),
        # instruction tuning of a 1B-class model on packed conversations: documents of
        # unequal lengths in one row, whose total is no multiple of anything
        _train("train_1b_packed", batch=1, seq=6001, hidden=2048, inter=8192, layers=3, heads=16,
               kv_heads=8, packed=9),
        # the headline: full fine-tuning of Llama-3-8B at sequence length 4096
        _train("train_8b", batch=2, seq=4096, hidden=4096, inter=14336, layers=4, heads=32,
               kv_heads=8, fused=True),
        # the same model with rank-32 adapters on every projection, base frozen
        _train("train_8b_lora", batch=2, seq=4096, hidden=4096, inter=14336, layers=3, heads=32,
               kv_heads=8, fused=True, rank=32),
        # attention of a long-context step
        _attn("attn_16k", batch=1, seq=16384, heads=32, kv_heads=8, dqk=128, dv=128),
        # latent (MLA) attention as it trains: 128 + 64 query/key columns, odd length
        _attn("attn_mla", batch=2, seq=3001, heads=16, kv_heads=16, dqk=192, dv=128),
        # the expert layer of Qwen3-30B-A3B
        _moe("moe_128x8", batch=2, seq=4096, hidden=2048, inter=768, experts=128, active=8),
        # a DeepSeek-style expert layer: sigmoid scores, a routing bias, shared experts; few,
        # odd tokens, as under expert parallelism or in short batches
        _moe("moe_64x6_shared", batch=3, seq=1001, hidden=2048, inter=1408, experts=64, active=6,
             shared=2816, sigmoid=True),
        # one conversation: short prompt, then token by token
        _gen("gen_llama_b1", model="llama", batch=1, prompt=511, ragged=False, new=32, hidden=4096,
             inter=14336, layers=4, heads=32, kv_heads=8),
        # a batch of equal prompts at an ordinary context
        _gen("gen_llama_b16", model="llama", batch=16, prompt=1500, ragged=False, new=32,
             hidden=4096, inter=14336, layers=4, heads=32, kv_heads=8),
        # one conversation with the latent-attention model
        _gen("gen_rezadra_b1", model="rezadra", batch=1, prompt=200, ragged=True, new=32,
             hidden=2048, inter=9216, layers=4, heads=16),
        # requests of unequal lengths packed together
        _gen("gen_rezadra_b8", model="rezadra", batch=8, prompt=1500, ragged=True, new=32,
             hidden=4096, inter=21504, layers=4, heads=32),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "packed", "lora", "attn", "moe", "gen_llama", "gen_rezadra"])
    if kind in ("train", "packed", "lora"):
        heads = rng.choice([2, 4, 8, 12, 16, 20, 32])
        kv = rng.choice([k for k in (1, 2, 4, 8, 16, 32) if heads % k == 0 and heads // k <= 8])
        tokens = _log(rng, 200, 8000)
        batch = 1 if kind == "packed" else rng.choice([b for b in (1, 2, 3, 4) if tokens // b >= 100])
        seq = min(tokens // batch, 4096)
        if rng.random() < 0.5:
            seq = max(128, seq // 128 * 128)
        hidden = heads * 128
        return _train(batch=batch, seq=seq, hidden=hidden, inter=int(hidden * rng.choice([2, 3.5, 4])),
                      layers=rng.choice([1, 2, 3]), heads=heads, kv_heads=kv,
                      vocab=rng.choice([1024, 32000, VOCAB]), fused=rng.random() < 0.5,
                      packed=rng.randint(2, 16) if kind == "packed" else 0,
                      rank=rng.choice([8, 32, 64]) if kind == "lora" else 0)
    if kind == "attn":
        dqk, dv = rng.choice([(64, 64), (96, 96), (128, 128), (128, 128), (192, 128), (192, 128),
                              (256, 256), (80, 80)])
        seq = _log(rng, 100, 16000)
        heads = rng.choice([4, 8, 14, 16, 32])
        kv = heads if dqk == 192 else rng.choice([k for k in (2, 4, 8, 14, 16, 32) if heads % k == 0])
        batch = rng.choice([b for b in (1, 2, 3, 4, 8) if b == 1 or b * heads * seq * seq < 2e9])
        return _attn(batch=batch, seq=seq, heads=heads, kv_heads=kv, dqk=dqk, dv=dv)
    if kind == "moe":
        experts, active = rng.choice([(8, 2), (32, 4), (64, 6), (128, 8)])
        sigmoid = rng.random() < 0.5
        return _moe(batch=rng.choice([1, 2, 3]), seq=_log(rng, 60, 2700),
                    hidden=rng.choice([1024, 2048]), inter=rng.choice([512, 768, 1408]),
                    experts=experts, active=active, shared=rng.choice([0, 1024, 2816]),
                    sigmoid=sigmoid)
    heads = rng.choice([8, 16, 32])
    hidden, batch = heads * 128, rng.choice([1, 2, 4, 7, 12, 16])
    if kind == "gen_llama":
        return _gen(model="llama", batch=batch, prompt=_log(rng, 20, 1500), ragged=False,
                    new=rng.choice([8, 16, 32]), hidden=hidden, inter=int(hidden * 3.5),
                    layers=rng.choice([2, 4]), heads=heads, kv_heads=rng.choice([4, 8]))
    return _gen(model="rezadra", batch=batch, prompt=_log(rng, 20, 1500), ragged=True,
                new=rng.choice([8, 16, 32]), hidden=hidden, inter=int(hidden * 4.5),
                layers=4, heads=heads)


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------

def _gen_of(seed):
    return torch.Generator(device=DEV).manual_seed(seed * 7919 + 13)


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32).mul_(std).to(BF)


def _doc_lengths(total, n, seed):
    """n unequal document lengths that add up to total."""
    r = torch.Generator().manual_seed(seed * 31 + 7)
    cuts = torch.randperm(total - 1, generator=r)[: n - 1].sort().values + 1
    edges = [0, *cuts.tolist(), total]
    return [b - a for a, b in zip(edges, edges[1:])]


def _llama_shapes(c):
    H, D = c["hidden"], c["head_dim"]
    q, kv, inter = c["heads"] * D, c["kv_heads"] * D, c["inter"]
    shapes = {"model.embed_tokens.weight": (c["vocab"], H), "model.norm.weight": (H,),
              "lm_head.weight": (c["vocab"], H)}
    for i in range(c["layers"]):
        p = f"model.layers.{i}."
        if c["fused"]:
            lin = {"self_attn.qkv_proj": (q + 2 * kv, H), "mlp.gate_up_proj": (2 * inter, H)}
        else:
            lin = {"self_attn.q_proj": (q, H), "self_attn.k_proj": (kv, H),
                   "self_attn.v_proj": (kv, H), "mlp.gate_proj": (inter, H),
                   "mlp.up_proj": (inter, H)}
        lin |= {"self_attn.o_proj": (H, q), "mlp.down_proj": (H, inter)}
        for n, (o, k) in lin.items():
            if c["rank"]:
                shapes[f"{p}{n}.base.weight"] = (o, k)
                shapes[f"{p}{n}.lora_A.weight"] = (c["rank"], k)
                shapes[f"{p}{n}.lora_B.weight"] = (o, c["rank"])
            else:
                shapes[f"{p}{n}.weight"] = (o, k)
        shapes[p + "input_layernorm.weight"] = (H,)
        shapes[p + "post_attention_layernorm.weight"] = (H,)
    return shapes


def _rezadra_shapes(c):
    W, h = c["hidden"], c["heads"]
    shapes = {"model.embed_tokens.weight": (c["vocab"], W), "model.embed_norm.weight": (W,),
              "model.loop_input.proj.weight": (W, 2 * W), "model.norm.weight": (W,),
              "lm_head.weight": (c["vocab"], W)}
    for i in range(c["layers"]):
        p = f"model.layers.{i}."
        shapes |= {p + "self_attn.q_kv_a_proj.weight": (h * 192 + 576, W),
                   p + "self_attn.kv_a_layernorm.weight": (512,),
                   p + "self_attn.kv_b_proj.weight": (h * 256, 512),
                   p + "self_attn.o_proj.weight": (W, h * 128),
                   p + "mlp.up_proj.weight": (c["inter"], W),
                   p + "mlp.down_proj.weight": (W, c["inter"])}
        for n in ("input", "post_attention", "pre_feedforward", "post_feedforward"):
            shapes[f"{p}{n}_layernorm.weight"] = (W,)
    return shapes


def _weights(shapes, seed):
    """Weights of a model under way: every projection keeps the size of what it is given (std
    fan-in^-1/2), embeddings and norms of about 1, adapters that have learnt."""
    g, out = _gen_of(seed), {}
    for n, s in shapes.items():
        if len(s) == 1:
            out[n] = (1 + 0.1 * torch.randn(s, generator=g, device=DEV)).to(BF)
        elif "lora_A" in n:
            out[n] = _randn(g, *s, std=1 / math.sqrt(3 * s[1]))
        elif "lora_B" in n:
            out[n] = _randn(g, *s, std=0.01)
        else:
            out[n] = _randn(g, *s, std=1.0 if "embed" in n else 1 / math.sqrt(s[1]))
    return out


def _load(model, weights):
    with torch.no_grad():
        mine = dict(model.named_parameters())
        assert set(mine) == set(weights), sorted(set(mine) ^ set(weights))
        for n, p in mine.items():
            p.copy_(weights[n])


def _llama_config(c, positions):
    return dict(vocab_size=c["vocab"], hidden_size=c["hidden"], intermediate_size=c["inter"],
                num_hidden_layers=c["layers"], num_attention_heads=c["heads"],
                num_key_value_heads=c["kv_heads"], head_dim=128, rope_theta=500000.0,
                rms_norm_eps=1e-5, max_position_embeddings=positions)


def _rezadra_config(c):
    return dict(vocab_size=c["vocab"], hidden_size=c["hidden"], num_hidden_layers=c["layers"],
                loop={"start": 1, "stop": 3, "times": 2}, num_attention_heads=c["heads"],
                intermediate_size=c["inter"], residual_multiplier=0.5, kv_lora_rank=512,
                qk_nope_head_dim=128, qk_rope_head_dim=64, v_head_dim=128)


def _tokens(c, seed):
    g = _gen_of(seed + 1_000_003)
    ids = torch.randint(0, c["vocab"], (c["batch"], c["seq"] + 1), generator=g, device=DEV)
    labels = ids[:, 1:].clone()
    labels[:, : c["seq"] // 8] = -100                       # a prompt that is not trained on
    return ids[:, :-1].clone(), labels


def _prompts(c, seed):
    r = torch.Generator().manual_seed(seed * 17 + 3)
    lens = [c["prompt"]] * c["batch"]
    if c["ragged"] and c["batch"] > 1:
        lens = torch.randint(max(1, c["prompt"] // 10), c["prompt"] + 1, (c["batch"],),
                             generator=r).tolist()
    prompts = [torch.randint(0, VOCAB, (n,), generator=r).tolist() for n in lens]
    return prompts, torch.randint(0, VOCAB, (c["new"], c["batch"]), generator=r)


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------

def prepare(case, seed):
    c = dict(case)
    if c["kind"] == "train":
        return _prepare_train(c, seed)
    if c["kind"] == "gen":
        return _prepare_gen(dict(c, vocab=VOCAB, head_dim=128, fused=False, rank=0), seed)
    if c["kind"] == "attn":
        q, k, v, do = _attn_inputs(c, seed)
        return dict(kind="attn", qkv=[t.requires_grad_() for t in (q, k, v)], do=do)
    from automodel_amd.moe.config import MoEConfig
    from automodel_amd.moe.layers import MoE

    cfg = MoEConfig(n_routed_experts=c["experts"], n_activated_experts=c["active"],
                    moe_intermediate_size=c["inter"], n_shared_experts=2 if c["shared"] else 0,
                    shared_expert_intermediate_size=c["shared"] or None,
                    score_func="sigmoid" if c["sigmoid"] else "softmax",
                    expert_bias=c["sigmoid"], route_scale=2.5 if c["sigmoid"] else 1.0)
    with torch.device("meta"):
        moe = MoE(c["hidden"], cfg)
    moe = moe.to(BF).to_empty(device=DEV)
    weights, bias, x, dy = _moe_inputs(c, seed)
    _load(moe, weights)
    if bias is not None:
        moe.gate.e_score_correction_bias.copy_(bias)
    return dict(kind="moe", moe=moe, x=x.requires_grad_(), dy=dy)


def _prepare_train(c, seed):
    from automodel_amd.loss.linear_ce import FusedLinearCrossEntropy
    from automodel_amd.models.common.backend import BackendConfig
    from automodel_amd.models.llama.model import LlamaConfig, LlamaForCausalLM
    from automodel_amd.optim.adamw import FusedAdamW
    from automodel_amd.peft.lora import PeftConfig, apply_lora_to_linear_modules

    cfg = LlamaConfig(**_llama_config(c, 8192), fused_qkv=c["fused"], fused_gate_up=c["fused"])
    with torch.device("meta"):
        model = LlamaForCausalLM(cfg, backend=BackendConfig(attn="hip", loss="hybrid"))
    model = model.to(BF)
    model.loss_fn = FusedLinearCrossEntropy(backend="hybrid", chunk_size=4096)
    if c["rank"]:
        apply_lora_to_linear_modules(model, PeftConfig(
            target_modules=["*_proj"], dim=c["rank"], alpha=2.0 * c["rank"]))
    model.init_weights(device=DEV)
    _load(model, _weights(_llama_shapes(c), seed))
    model.train()
    params = {n: p for n, p in model.named_parameters() if p.requires_grad}
    opt = FusedAdamW(list(params.values()), lr=2e-5, weight_decay=0.0)
    ids, labels = _tokens(c, seed)
    cu = pos = None
    if c["packed"]:
        lens = _doc_lengths(c["seq"], c["packed"], seed)
        cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32).to(DEV)
        pos = torch.cat([torch.arange(n) for n in lens]).unsqueeze(0).to(DEV)
    return dict(kind="train", model=model, opt=opt, params=params, ids=ids, labels=labels, cu=cu,
                pos=pos)


def _prepare_gen(c, seed):
    from automodel_amd.models.registry import build_model
    from automodel_amd.serving import swap_linears_for_decode
    from automodel_amd.utils.generation import DecodeSession

    llama = c["model"] == "llama"
    model = build_model(config=_llama_config(c, 4096) if llama else _rezadra_config(c),
                        architecture="LlamaForCausalLM" if llama else "Rezadra",
                        dtype="bfloat16", meta_init=True)
    model.init_weights(device=DEV)
    _load(model, _weights(_llama_shapes(c) if llama else _rezadra_shapes(c), seed))
    model.eval()
    if llama and c["batch"] <= 4:
        swap_linears_for_decode(model)
    prompts, more = _prompts(c, seed)
    session = DecodeSession(model, c["batch"], c["prompt"] + c["new"])
    return dict(kind="gen", session=session, prompts=prompts, more=more.to(DEV))


def run(state):
    kind = state["kind"]
    if kind == "attn":
        from automodel_amd.ops.attention import flash_attention

        q, k, v = state["qkv"]
        o = flash_attention(q, k, v, causal=True)
        dq, dk, dv = torch.autograd.grad(o, (q, k, v), state["do"])
        return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv}
    if kind == "moe":
        moe, x = state["moe"], state["x"]
        params = dict(moe.named_parameters())
        y = moe(x)
        grads = torch.autograd.grad(y, [x, *params.values()], state["dy"])
        return {"y": y.detach(), "dx": grads[0], "grad": dict(zip(params, grads[1:]))}
    if kind == "train":
        return _train_step(state)
    # a greedy loop as generate_cached has it, but scoring a given continuation
    session = state["session"]
    handles, logits = session.prefill(state["prompts"])
    out = [logits]
    for tokens in state["more"]:
        out.append(session.decode(handles, tokens))
    session.release(handles)
    return {"logits": torch.stack(out, dim=1)}


def _train_step(state):
    from automodel_amd.ops.attention import set_varlen_context

    model, opt, labels = state["model"], state["opt"], state["labels"]
    opt.zero_grad(set_to_none=True)
    set_varlen_context(state["cu"])
    try:
        loss = model(state["ids"], labels=labels, position_ids=state["pos"])
        (loss / labels.numel()).backward()
    finally:
        set_varlen_context(None)
    opt.step()
    params = state["params"]
    return {"loss": loss.detach(), "grad": {n: p.grad for n, p in params.items()},
            "weight": {n: p.detach() for n, p in params.items()}}


def _attn_inputs(c, seed):
    g = _gen_of(seed)
    B, S, H, K = c["batch"], c["seq"], c["heads"], c["kv_heads"]
    return (_randn(g, B, S, H, c["dqk"]), _randn(g, B, S, K, c["dqk"]),
            _randn(g, B, S, K, c["dv"]), _randn(g, B, S, H, c["dv"]))


def _moe_inputs(c, seed):
    E, H, I, S = c["experts"], c["hidden"], c["inter"], c["shared"]
    shapes = {"gate.weight": (E, H), "experts.gate_proj": (E, I, H), "experts.up_proj": (E, I, H),
              "experts.down_proj": (E, H, I)}
    if S:
        shapes |= {"shared_experts.gate_proj.weight": (S, H),
                   "shared_experts.up_proj.weight": (S, H),
                   "shared_experts.down_proj.weight": (H, S)}
    g = _gen_of(seed)
    weights = {n: _randn(g, *s, std=0.02) for n, s in shapes.items()}
    bias = _randn(g, E, std=0.02) if c["sigmoid"] else None
    x = _randn(g, c["batch"], c["seq"], H)
    return weights, bias, x, _randn(g, c["batch"], c["seq"], H)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _pairs(lens):
    return sum(n * (n + 1) // 2 for n in lens)


def work(case):
    c = dict(case)
    if c["kind"] == "attn":
        B, S, H, K, dq, dv = (c[k] for k in ("batch", "seq", "heads", "kv_heads", "dqk", "dv"))
        qo, kv = B * S * H * (dq + dv) * 2, B * S * K * (dq + dv) * 2
        # forward S = QK, O = PV; backward S, dP, dV, dQ, dK
        flops = 2 * B * H * _pairs([S]) * (4 * dq + 3 * dv)
        return {"bytes": 2 * qo + 2 * kv, "flops": flops}
    if c["kind"] == "moe":
        T, E, k, H, I, S = c["batch"] * c["seq"], *(c[n] for n in ("experts", "active", "hidden",
                                                                   "inter", "shared"))
        params = E * H + 3 * E * H * I + 3 * H * S
        return {"bytes": 2 * (2 * params + 4 * T * H),
                "flops": 6 * T * (E * H + 3 * H * (k * I + S))}
    if c["kind"] == "train":
        shapes = _llama_shapes(c)
        T = c["batch"] * c["seq"]
        lin = sum(math.prod(s) for n, s in shapes.items()
                  if len(s) == 2 and "embed" not in n and "lora" not in n)
        ad = sum(math.prod(s) for n, s in shapes.items() if "lora" in n)
        lens = [c["seq"]] * c["batch"] if not c["packed"] else _doc_lengths(c["seq"], c["packed"], 1)
        attn = c["layers"] * c["heads"] * c["head_dim"] * _pairs(lens)
        total = sum(math.prod(s) for s in shapes.values())
        if c["rank"]:       # frozen base: no weight gradients; adapters have optimizer state
            return {"bytes": 2 * total + 28 * ad, "flops": T * (4 * lin + 6 * ad) + 14 * attn}
        return {"bytes": 2 * total + 30 * total, "flops": 6 * T * lin + 14 * attn}
    c |= dict(vocab=VOCAB, head_dim=128, fused=False, rank=0)
    prompts, _ = _prompts(c, 1)
    n, T, new = c["batch"], sum(map(len, prompts)), c["new"]
    shapes = _llama_shapes(c) if c["model"] == "llama" else _rezadra_shapes(c)
    runs = [1] * c["layers"] if c["model"] == "llama" else [1, 2, 2, 1]
    lin = sum(math.prod(s) * (runs[int(k.split(".")[2])] if ".layers." in k else 1)
              for k, s in shapes.items() if len(s) == 2 and "embed" not in k and "lm_head" not in k)
    if "model.loop_input.proj.weight" in shapes:
        lin += math.prod(shapes["model.loop_input.proj.weight"])
    head = VOCAB * c["hidden"]
    row = sum(runs) * 2 * (2 * c["kv_heads"] * 128 if c["model"] == "llama" else 576)
    width = 256 if c["model"] == "llama" else 320
    seen = sum(sum(len(p) + j for j in range(1, new + 1)) for p in prompts)
    return {"bytes": 2 * (lin + head) * (1 + new) + row * (T + seen) + 4 * n * (new + 1) * VOCAB,
            "flops": 2 * lin * (T + n * new) + 2 * head * n * (new + 1)
            + 2 * sum(runs) * c["heads"] * width * (_pairs(map(len, prompts)) + seen)}


def tolerance(case):
    # bf16 in and out, sums in 32 bits. Measured against 64 bits: attention 0.0025, expert layers
    # 0.005, rezadra's logits (its residual is 32 bits) 0.004, llama's logits 0.01, gradients
    # through whole models 0.013; another order of the sums moves those by up to 0.01. About four
    # times that, at most 0.03
    if case["kind"] == "attn":
        return {"rel": 0.01, "max": 0.4}
    if case["kind"] == "moe" or case.get("model") == "rezadra":
        return {"rel": 0.02, "max": 0.8}
    return {"rel": 0.03, "max": 0.9}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def exact(case, seed):
    c = dict(case)
    if c["kind"] == "attn":
        return _exact_attn(c, seed)
    if c["kind"] == "moe":
        return _exact_moe(c, seed)
    if c["kind"] == "train":
        return _exact_train(c, seed)
    return _exact_gen(dict(c, vocab=VOCAB, head_dim=128, fused=False, rank=0), seed)


def _causal(n):
    return torch.ones(n, n, dtype=torch.bool, device=DEV).tril_()


def _exact_attn(c, seed):
    q, k, v, do = (t.double() for t in _attn_inputs(c, seed))
    scale, G = 1 / math.sqrt(c["dqk"]), c["heads"] // c["kv_heads"]
    o, dq = torch.empty_like(do), torch.empty_like(q)
    dk, dv = torch.zeros_like(k), torch.zeros_like(v)
    keep = _causal(c["seq"])
    for b in range(c["batch"]):
        for h in range(c["heads"]):
            j = h // G
            qh, kh, vh, doh = q[b, :, h], k[b, :, j], v[b, :, j], do[b, :, h]
            p = (qh @ kh.T).mul_(scale).masked_fill_(~keep, -math.inf).softmax(-1)
            o[b, :, h] = oh = p @ vh
            dv[b, :, j] += p.T @ doh
            ds = (doh @ vh.T).sub_((doh * oh).sum(-1, keepdim=True)).mul_(p).mul_(scale)
            dq[b, :, h] = ds @ kh
            dk[b, :, j] += ds.T @ qh
    return {"o": o, "dq": dq, "dk": dk, "dv": dv}


def _silu_mul(g, u):
    return torch.nn.functional.silu(g) * u


def _exact_moe(c, seed):
    weights, bias, x, dy = _moe_inputs(c, seed)
    w = {n: t.double().requires_grad_() for n, t in weights.items()}
    x = x.double().requires_grad_()
    xf = x.reshape(-1, c["hidden"])
    logits = xf @ w["gate.weight"].T
    scores = logits.sigmoid() if c["sigmoid"] else logits.softmax(-1)
    pick = (scores + bias.double() if c["sigmoid"] else scores).topk(c["active"], -1)[1]
    probs = scores.gather(1, pick)
    probs = probs / probs.sum(-1, keepdim=True) * (2.5 if c["sigmoid"] else 1.0)
    y = torch.zeros_like(xf)
    for e in range(c["experts"]):
        rows, slot = (pick == e).nonzero(as_tuple=True)
        xe = xf[rows]
        h = _silu_mul(xe @ w["experts.gate_proj"][e].T, xe @ w["experts.up_proj"][e].T)
        y = y.index_add(0, rows, h @ w["experts.down_proj"][e].T * probs[rows, slot, None])
    if c["shared"]:
        h = _silu_mul(xf @ w["shared_experts.gate_proj.weight"].T,
                      xf @ w["shared_experts.up_proj.weight"].T)
        y = y + h @ w["shared_experts.down_proj.weight"].T
    y = y.view_as(x)
    grads = torch.autograd.grad(y, [x, *w.values()], dy.double())
    return {"y": y.detach(), "dx": grads[0], "grad": dict(zip(w, grads[1:]))}


def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope(x, pos, base):
    """x [..., T, heads, n], pairs (i, i + n/2) turned by pos * base^(-2i/n)."""
    n = x.shape[-1]
    f = base ** (-torch.arange(0, n, 2, device=DEV, dtype=torch.float64) / n)
    a = (pos.double()[:, None] * f).unsqueeze(-2)
    u, v = x[..., : n // 2], x[..., n // 2:]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1)


def _attend(q, k, v, scale):
    """One sequence: q [T, H, d], k/v [T, K, d] -> [T, H, dv]."""
    G = q.shape[1] // k.shape[1]
    k, v = (t.repeat_interleave(G, 1).permute(1, 0, 2) for t in (k, v))
    s = (q.permute(1, 0, 2) @ k.transpose(1, 2)) * scale
    p = s.masked_fill(~_causal(q.shape[0]), -math.inf).softmax(-1)
    return (p @ v).permute(1, 0, 2)


def _llama_hidden(c, w, ids, parts):
    """ids [T]; parts: the lengths of the sequences that lie in it, one after another."""
    from torch.utils.checkpoint import checkpoint

    H, K, D, I = c["heads"], c["kv_heads"], c["head_dim"], c["inter"]
    pos = torch.cat([torch.arange(n, device=DEV) for n in parts])

    def lin(x, n):
        if not c["rank"]:
            return x @ w[n + ".weight"].T
        y = x @ w[n + ".base.weight"].T
        return y + (x @ w[n + ".lora_A.weight"].T) @ w[n + ".lora_B.weight"].T * 2.0

    x = w["model.embed_tokens.weight"][ids]
    for i in range(c["layers"]):
        p = f"model.layers.{i}."
        h = _rms(x, w[p + "input_layernorm.weight"], 1e-5)
        if c["fused"]:
            q, k, v = lin(h, p + "self_attn.qkv_proj").split([H * D, K * D, K * D], -1)
        else:
            q, k, v = (lin(h, f"{p}self_attn.{n}_proj") for n in "qkv")
        q, k = (_rope(t.reshape(-1, n, D), pos, 500000.0) for t, n in ((q, H), (k, K)))
        o = [checkpoint(_attend, *t, D ** -0.5, use_reentrant=False)
             for t in zip(q.split(parts), k.split(parts), v.reshape(-1, K, D).split(parts))]
        x = x + lin(torch.cat(o).reshape(-1, H * D), p + "self_attn.o_proj")
        h = _rms(x, w[p + "post_attention_layernorm.weight"], 1e-5)
        if c["fused"]:
            g, u = lin(h, p + "mlp.gate_up_proj").split(I, -1)
        else:
            g, u = lin(h, p + "mlp.gate_proj"), lin(h, p + "mlp.up_proj")
        x = x + lin(_silu_mul(g, u), p + "mlp.down_proj")
    return _rms(x, w["model.norm.weight"], 1e-5)


def _exact_train(c, seed):
    w = {n: t.double() for n, t in _weights(_llama_shapes(c), seed).items()}
    live = {n: t.requires_grad_() for n, t in w.items() if not c["rank"] or "lora" in n}
    ids, labels = _tokens(c, seed)
    parts = _doc_lengths(c["seq"], c["packed"], seed) if c["packed"] else [c["seq"]] * c["batch"]
    hidden = _llama_hidden(c, w, ids.reshape(-1), parts)
    logits = hidden @ w["lm_head.weight"].T
    loss = torch.nn.functional.cross_entropy(logits, labels.reshape(-1), ignore_index=-100,
                                             reduction="sum")
    grads = dict(zip(live, torch.autograd.grad(loss / labels.numel(), list(live.values()))))
    # the first step of AdamW from zero moments
    weight = {n: (p - 2e-5 * grads[n] / (grads[n].abs() + 1e-8)).detach() for n, p in live.items()}
    return {"loss": loss.detach(), "grad": grads, "weight": weight}


def _rezadra_hidden(c, w, ids):
    W, H, eps, m = c["hidden"], c["heads"], 1e-6, 0.5
    pos = torch.arange(len(ids), device=DEV)
    x0 = x = _rms(w["model.embed_tokens.weight"][ids], w["model.embed_norm.weight"], eps)
    for i, begins in [(0, False), (1, True), (2, False), (1, True), (2, False), (3, False)]:
        p = f"model.layers.{i}."
        if begins:
            x = torch.cat([x, x0], -1) @ w["model.loop_input.proj.weight"].T
        h = _rms(x, w[p + "input_layernorm.weight"], eps)
        q, lat, kr = (h @ w[p + "self_attn.q_kv_a_proj.weight"].T).split([H * 192, 512, 64], -1)
        lat = _rms(lat, w[p + "self_attn.kv_a_layernorm.weight"], eps)
        kn, v = (lat @ w[p + "self_attn.kv_b_proj.weight"].T).split(H * 128, -1)
        q = q.view(-1, H, 192)
        q = torch.cat([q[..., :128], _rope(q[..., 128:], pos, 10000.0)], -1)
        kr = _rope(kr.unsqueeze(1), pos, 10000.0).expand(-1, H, -1)
        o = _attend(q, torch.cat([kn.view(-1, H, 128), kr], -1), v.view(-1, H, 128), 192 ** -0.5)
        y = o.reshape(-1, H * 128) @ w[p + "self_attn.o_proj.weight"].T
        x = x + m * _rms(y, w[p + "post_attention_layernorm.weight"], eps)
        h = _rms(x, w[p + "pre_feedforward_layernorm.weight"], eps)
        y = (h @ w[p + "mlp.up_proj.weight"].T).relu().square() @ w[p + "mlp.down_proj.weight"].T
        x = x + m * _rms(y, w[p + "post_feedforward_layernorm.weight"], eps)
    return _rms(x, w["model.norm.weight"], eps)


@torch.no_grad()
def _exact_gen(c, seed):
    llama = c["model"] == "llama"
    w = {n: t.double() for n, t in
         _weights(_llama_shapes(c) if llama else _rezadra_shapes(c), seed).items()}
    prompts, more = _prompts(c, seed)
    out = []
    for i, prompt in enumerate(prompts):
        ids = torch.tensor(prompt + more[:, i].tolist(), device=DEV)
        h = _llama_hidden(c, w, ids, [len(ids)]) if llama else _rezadra_hidden(c, w, ids)
        out.append(h[len(prompt) - 1:] @ w["lm_head.weight"].T)
    return {"logits": torch.stack(out)}
