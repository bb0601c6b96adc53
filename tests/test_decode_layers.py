"""Decode layers issued by one native call against the same layers module by module."""

import pytest
import torch

from automodel_amd.models.registry import build_model
from automodel_amd.utils.generation import DecodeSession

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def steps(model, batch, prompt_len, new):
    g = torch.Generator().manual_seed(0)
    prompts = torch.randint(0, 256, (batch, prompt_len), generator=g).tolist()
    more = torch.randint(0, 256, (new, batch), generator=g).cuda()
    session = DecodeSession(model, batch, prompt_len + new)
    handles, logits = session.prefill(prompts)
    return torch.stack([logits, *(session.decode(handles, t) for t in more)]), session.cache


def compare(model, modules, batch, monkeypatch, op, expected):
    from automodel_amd.ops._backend import hip_ops

    calls = []
    inner = getattr(hip_ops(), op)
    monkeypatch.setattr(hip_ops(), op, lambda *a: (calls.append(len(r := inner(*a))), r)[1])
    got, cache = steps(model, batch, 5, 4)
    assert (sum(calls) > 0) == expected
    for m in modules(model):                    # observed modules are called one by one
        m.register_forward_hook(lambda *a: None)
    calls.clear()
    want, ref_cache = steps(model, batch, 5, 4)
    assert not calls
    # both round to 8 bits after every kernel, at different places for the residual
    err = (got.float() - want.float()).norm() / want.float().norm()
    assert err < 2.0 ** -8 * 4, float(err)
    return cache, ref_cache


LLAMA = dict(vocab_size=256, hidden_size=256, intermediate_size=520, num_hidden_layers=3,
             num_attention_heads=4, num_key_value_heads=2, max_position_embeddings=64)


@pytest.mark.parametrize("batch", [1, 2, 3, 17, 32, 33])
@pytest.mark.parametrize("options,native", [
    ({}, True), (dict(fused_qkv=True, fused_gate_up=True), True), (dict(head_dim=96), True),
    (dict(tie_word_embeddings=True, logits_scaling=2.0, attention_multiplier=0.05), True),
    (dict(attention_bias=True), False), (dict(qk_norm=True), False), (dict(mlp_bias=True), False),
    (dict(residual_multiplier=0.5), False), (dict(olmo2_layout=True), False),
    (dict(rope_interleaved=True), False), (dict(intermediate_size=516), False),
])
def test_llama(batch, options, native, monkeypatch):
    if batch * options.get("intermediate_size", 8) % 8:
        pytest.skip("the activation kernel refuses the size")
    torch.manual_seed(0)
    model = build_model(config={**LLAMA, **options}, architecture="LlamaForCausalLM",
                        dtype="bfloat16", meta_init=True)
    model.init_weights(device="cuda")
    model.eval()
    cache, ref = compare(model, lambda m: [x.mlp for x in m.model.layers], batch, monkeypatch,
                         "llama_decode_layer", native and batch <= 32)
    assert cache.pos == ref.pos == 9
    for a, b in ((cache.k, ref.k), (cache.v, ref.v)):
        assert (a.float() - b.float()).norm() <= 2.0 ** -8 * 4 * b.float().norm()


@pytest.mark.parametrize("batch", [1, 2, 9, 17, 64, 65])
@pytest.mark.parametrize("width,inter,heads,rank", [(256, 512, 4, 64), (512, 776, 3, 512), (256, 510, 4, 64)])
def test_latent(batch, width, inter, heads, rank, monkeypatch):
    torch.manual_seed(0)
    model = build_model(config=dict(
        vocab_size=256, hidden_size=width, num_hidden_layers=3, num_attention_heads=heads,
        intermediate_size=inter, residual_multiplier=0.5, kv_lora_rank=rank, qk_nope_head_dim=64,
        qk_rope_head_dim=32, v_head_dim=64, loop={"start": 1, "stop": 2, "times": 2}),
        architecture="Rezadra", dtype="bfloat16", meta_init=True)
    model.init_weights(device="cuda")
    model.eval()
    compare(model, lambda m: [x.self_attn for x in m.model.layers], batch, monkeypatch,
            "latent_decode_layer", batch <= 64 and inter % 8 == 0)
