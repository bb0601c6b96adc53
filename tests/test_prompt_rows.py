"""Which tokens' logits a prompt on the dense K/V cache returns."""

import pytest
import torch

from automodel_amd.models.registry import build_model
from automodel_amd.utils.generation import DecodeSession

PROMPTS = [[5, 6, 7], [8, 9, 10]]


@pytest.fixture(scope="module")
def model():
    torch.manual_seed(0)
    m = build_model(config=dict(vocab_size=64, hidden_size=32, intermediate_size=64, num_hidden_layers=1,
                                num_attention_heads=2, num_key_value_heads=1, head_dim=16,
                                max_position_embeddings=32), dtype="float32", meta_init=True)
    m.init_weights(device="cpu")
    return m.eval()


@pytest.mark.parametrize("want", [[[], []], [[], [1]], [[0, 2], []], [[-1, 0], [2, -3]]])
def test_wanted_rows(model, want):
    _, logits = DecodeSession(model, 2, 8).prefill(PROMPTS, want)
    with torch.no_grad():
        full = model(torch.tensor(PROMPTS))
    # a product of fewer rows may sum in another order: 32 terms of size below 1, in float32
    torch.testing.assert_close(logits, torch.cat([full[i, w] for i, w in enumerate(want)]),
                               rtol=0, atol=32 * 2.0 ** -23)


@pytest.mark.parametrize("want", [[[3], [0]], [[5], [1]], [[0], [1, -4]], [[0], [1], [2]]])
def test_rows_beyond_the_prompt_are_refused(model, want):
    session = DecodeSession(model, 2, 8)
    with pytest.raises(IndexError):
        session.prefill(PROMPTS, want)
    assert session.live == [] and session.cache.pos == 0
