"""Linear cross-entropy: logits kept for the backward or computed again, any number of chunks."""

import pytest
import torch

from automodel_amd.loss.linear_ce import FusedLinearCrossEntropy, _kept_chunks

gpu = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def test_kept_rows_fit_the_weight_gradient():
    for T in (1, 100, 4096, 4097, 9000, 100000):
        for H, V, chunk in ((256, 1024, 128), (2048, 32768, 4096), (4096, 128256, 4096), (64, 512, 4096)):
            n = _kept_chunks(T, H, V, chunk)
            assert 0 <= n <= -(-T // chunk) and 2 * n * chunk * V <= 4 * V * H


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("T", [1, 100, 128, 200, 256, 300, 700])
@pytest.mark.parametrize("train_weight,train_hidden", [(True, True), (False, True), (True, False)])
def test_same_gradients(T, train_weight, train_hidden):
    torch.manual_seed(0)
    H, V, chunk = 128, 1000, 128
    hidden = torch.randn(T, H, device="cuda").bfloat16()
    weight = torch.randn(V, H, device="cuda").bfloat16() * 0.1
    labels = torch.randint(0, V, (T,), device="cuda")
    labels[T // 2 :: 7] = -100
    results = []
    for keep in (True, False):
        h = hidden.clone().requires_grad_(train_hidden)
        w = weight.clone().requires_grad_(train_weight)
        loss = FusedLinearCrossEntropy("hybrid", chunk, keep_logits=keep)(h, w, labels)
        inputs = [t for t in (h, w) if t.requires_grad]
        first = torch.autograd.grad(loss / 3, inputs, retain_graph=True)
        again = torch.autograd.grad(loss / 3, inputs)
        for a, b in zip(first, again):
            assert torch.equal(a, b)
        results.append(first)
    for a, b in zip(*results):
        assert torch.equal(a, b)
    h, w = hidden.double().requires_grad_(train_hidden), weight.double().requires_grad_(train_weight)
    ref = torch.nn.functional.cross_entropy(h @ w.t(), labels, ignore_index=-100, reduction="sum")
    # logits, their gradient and the result are rounded to bf16: 2^-9 each, the logits' error
    # (of up to 4) entering through the exponential
    for a, b in zip(results[0], torch.autograd.grad(ref / 3, [t for t in (h, w) if t.requires_grad])):
        assert (a.double() - b).norm() <= (2 + 4) * 2.0 ** -9 * b.norm()
