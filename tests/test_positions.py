"""A decode step behind the last position of a model is refused where the host knows the position."""

import pytest
import torch

from automodel_amd.models.llama.model import LlamaConfig, LlamaForCausalLM
from automodel_amd.utils.generation import DecodeSession, generate_cached, generate_graphed

gpu = pytest.param("cuda", marks=[pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")])


def _model(device, **options):
    torch.manual_seed(0)
    model = LlamaForCausalLM(LlamaConfig(vocab_size=64, hidden_size=256, intermediate_size=256, num_hidden_layers=1,
                                         num_attention_heads=2, num_key_value_heads=1, head_dim=128,
                                         max_position_embeddings=8, **options))
    model.init_weights()
    return model.to(device, torch.bfloat16 if device == "cuda" else torch.float32).eval()


@pytest.mark.parametrize("device", ["cpu", gpu])
def test_the_last_position(device):
    model = _model(device)
    session = DecodeSession(model, 1, 12)
    handles, logits = session.prefill([[1, 2, 3, 4, 5, 6, 7]])
    logits = session.decode(handles, logits.argmax(-1))              # the eighth
    assert logits.isfinite().all()
    with pytest.raises(IndexError):
        session.decode(handles, logits.argmax(-1))
    prompt = torch.tensor([[1, 2, 3, 4, 5]], device=device)
    for f in (generate_cached, generate_graphed):
        assert f(model, prompt, 4).shape == (1, 9)                   # the ninth token is not looked at
        with pytest.raises(IndexError):
            f(model, prompt, 5)
    assert generate_graphed(model, torch.arange(8, device=device)[None], 1).shape == (1, 9)


def test_layers_without_positions():
    assert _model("cpu").model.positions == 8 and _model("cpu", no_rope_layers=[0]).model.positions is None
