"""One-token attention over the dense K/V cache, and the decode loop that uses it."""

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("B,H,K,D,length,pos", [
    (1, 4, 4, 64, 70, 0), (2, 8, 2, 128, 300, 299), (1, 32, 8, 128, 600, 511), (3, 14, 2, 80, 1000, 333),
    (2, 16, 2, 256, 130, 64), (1, 3, 1, 96, 129, 128), (130, 8, 8, 128, 80, 63), (1, 48, 2, 192, 5000, 4097),
    (1, 5, 1, 8, 40, 17),
])
@pytest.mark.parametrize("on_device", [False, True])
def test_against_f64(B, H, K, D, length, pos, on_device):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    q = torch.randn(B, 1, H, D, device="cuda").bfloat16() * 2
    kn, vn = (torch.randn(B, 1, K, D, device="cuda").bfloat16() for _ in range(2))
    kc, vc = (torch.randn(B, length, K, D, device="cuda").bfloat16() for _ in range(2))
    kc[:, pos:], vc[:, pos:] = float("nan"), float("nan")       # never read
    k0, v0 = kc.clone(), vc.clone()
    at = torch.tensor(pos, device="cuda") if on_device else None
    o = hip_ops().kv_decode_attn(q, kn, vn, kc, vc, -1 if on_device else pos, at, D ** -0.5)
    k0[:, pos], v0[:, pos] = kn[:, 0], vn[:, 0]
    assert torch.equal(kc.view(torch.int16), k0.view(torch.int16))
    assert torch.equal(vc.view(torch.int16), v0.view(torch.int16))
    kf, vf = (t[:, :pos + 1].double().repeat_interleave(H // K, 2).transpose(1, 2).contiguous()
              for t in (kc, vc))
    s = (kf @ q[:, 0].double()[..., None])[..., 0] * D ** -0.5
    ref = (s.softmax(-1)[:, :, None] @ vf)[:, :, 0]
    # f32 throughout; the output is rounded to bf16 once
    assert (o[:, 0].double() - ref).norm() <= 2.0 ** -9 * ref.norm() * 1.01


@pytest.mark.parametrize("heads,kv,dim", [(4, 2, 128), (6, 1, 64)])
def test_decode_matches_whole_forward(heads, kv, dim):
    """Prompt and one-token steps give the logits of one forward over all tokens."""
    from automodel_amd.models.registry import build_model
    from automodel_amd.utils.generation import DecodeSession, generate_graphed, generate_cached

    torch.manual_seed(0)
    model = build_model(config=dict(vocab_size=512, hidden_size=heads * dim, intermediate_size=512,
                                    num_hidden_layers=2, num_attention_heads=heads,
                                    num_key_value_heads=kv, head_dim=dim,
                                    max_position_embeddings=512), dtype="bfloat16", meta_init=True)
    model.init_weights(device="cuda")
    model.eval()
    ids = torch.randint(0, 512, (3, 150))
    session = DecodeSession(model, 3, 160)
    handles, logits = session.prefill(ids[:, :131].tolist(), want=[[130], [0, 130], [-1]])
    rows = [logits[[0, 2, 3]]]
    for j in range(131, 150):
        rows.append(session.decode(handles, ids[:, j].cuda()))
    with torch.no_grad():
        full = model(ids.cuda())
    got, want = torch.stack(rows, 1).float(), full[:, 130:].float()
    assert (got - want).norm() / want.norm() < 0.02     # a few bf16 roundings per layer
    first = full[1, 0].float()
    assert (logits[1].float() - first).norm() / first.norm() < 0.02
    prompt = ids[:, :20].cuda()
    eager = generate_graphed(model, prompt, 12, use_hip_graph=False)
    for _ in range(2):
        assert torch.equal(generate_graphed(model, prompt, 12), eager)
    assert torch.equal(generate_cached(model, prompt, 2), eager[:, :22])


@pytest.mark.parametrize("elsewhere", [1, 2, 3, 4, 5])
def test_tensors_elsewhere_are_refused(elsewhere):
    from automodel_amd.ops._backend import hip_ops

    args = [torch.zeros(1, 1, 2, 64, dtype=torch.bfloat16), torch.zeros(1, 1, 1, 64, dtype=torch.bfloat16),
            torch.zeros(1, 1, 1, 64, dtype=torch.bfloat16), torch.zeros(1, 9, 1, 64, dtype=torch.bfloat16),
            torch.zeros(1, 9, 1, 64, dtype=torch.bfloat16), torch.tensor(0)]
    args = [t if i == elsewhere else t.cuda() for i, t in enumerate(args)]
    with pytest.raises(RuntimeError):
        hip_ops().kv_decode_attn(*args[:5], -1, args[5], 0.125)
