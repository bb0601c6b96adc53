"""Shared experts on a stream of their own beside the routed ones: which modules are told so."""

import pytest
import torch

from automodel_amd.moe.config import MoEConfig
from automodel_amd.moe.layers import MoE, SharedExpert, _takes_beside


class Made(SharedExpert):
    """As sharding puts a class of its own in a module's place."""


class Other(SharedExpert):
    def forward(self, x):
        return 2 * super().forward(x)


def _kinds():
    """{name: (module, whether it is told, its output for its weights' by SharedExpert)}"""
    made = {n: cls(64, 128) for n, cls in (("plain", SharedExpert), ("made", Made), ("other", Other), ("replaced", SharedExpert))}
    forward = made["replaced"].forward
    made["replaced"].forward = lambda x: 2 * forward(x)
    return {n: (m, n in ("plain", "made"), 1 if n in ("plain", "made") else 2) for n, m in made.items()}


@pytest.mark.parametrize("kind", ["plain", "made", "other", "replaced"])
def test_who_is_told(kind):
    module, told, times = _kinds()[kind]
    assert _takes_beside(module) == told
    x = torch.randn(3, 64)
    assert torch.equal(module(x, **({"beside": True} if told else {})), times * SharedExpert.forward(module, x))


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("kind", ["plain", "made", "other", "replaced"])
def test_layer(kind):
    torch.manual_seed(0)
    cfg = MoEConfig(n_routed_experts=4, n_activated_experts=2, moe_intermediate_size=128, n_shared_experts=1)
    moe, (module, _, times) = MoE(64, cfg), _kinds()[kind]
    with torch.no_grad():
        for p in moe.parameters():
            p.normal_(std=0.1)
    moe.shared_experts = module
    moe = moe.to("cuda", torch.bfloat16)
    x = torch.randn(1, 5, 64, device="cuda").bfloat16()
    y = moe(x)
    moe.shared_experts = None
    shared = times * SharedExpert.forward(module, x.view(5, 64))
    # three roundings to 8 bits of either, each 2^-9 of a value at most
    assert (y - moe(x) - shared).abs().max() <= 6 * 2.0 ** -9 * max(float(y.abs().max()), float(shared.abs().max()))
