"""What a decode step begins with, in one launch (csrc/rope.hip: token_rows)."""

import pytest
import torch
import torch.nn as nn

from automodel_amd.ops.rope import token_rows

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def _inputs(W, D, dtype, vocab=37, places=50):
    torch.manual_seed(W)
    embed = nn.Embedding(vocab, W, device="cuda", dtype=torch.bfloat16)
    return embed, *(torch.randn(places, D, device="cuda").to(dtype) for _ in range(2))


# a part of a block, one, several and a remainder; both kinds of tables; the first and last row of each
@pytest.mark.parametrize("W,D", [(8, 2), (2048, 64), (2056, 128), (4104, 256)])
@pytest.mark.parametrize("B,S", [(1, 1), (64, 1), (3, 5)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows(W, D, B, S, dtype):
    embed, cos, sin = _inputs(W, D, dtype)
    ids = torch.randint(0, 37, (B, S), device="cuda")
    ids.view(-1)[0], ids.view(-1)[-1] = 0, 36
    pos = torch.arange(51, device="cuda")[50 - S:50] if S > 1 else torch.tensor([0], device="cuda")
    with torch.no_grad():
        x, c, s = token_rows(embed, ids, pos, cos, sin)
        assert torch.equal(x, embed(ids)) and torch.equal(c, cos[pos].float()) and torch.equal(s, sin[pos].float())
        _, c, s = token_rows(embed, ids, pos - 50, cos, sin)          # from the end
        assert torch.equal(c, cos[pos - 50].float()) and torch.equal(s, sin[pos - 50].float())


def test_what_is_none_and_what_is_left():
    embed, cos, sin = _inputs(64, 16, torch.bfloat16)
    ids, pos = torch.tensor([[3], [37], [-1]], device="cuda"), torch.tensor([50, 1, -51], device="cuda")
    with torch.no_grad():
        x, c, s = token_rows(embed, ids, pos, cos, sin)
        assert torch.equal(x[0], embed(ids[0])) and x[1:].isnan().all() and c[[0, 2]].isnan().all()
        assert torch.equal(c[1], cos[1].float()) and torch.equal(s[1], sin[1].float()) and s[[0, 2]].isnan().all()
        ids, pos = ids[:1], pos[1:2]
        for args in ((embed, ids.int(), pos, cos, sin), (embed, ids, pos.int(), cos, sin), (embed, ids, pos[0], cos, sin),
                     (embed, ids, pos, cos.half(), sin.half()), (embed, ids, pos, cos, sin.float()),
                     (embed, ids, pos, cos.t().contiguous().t(), sin), (embed.float(), ids, pos, cos, sin)):
            assert token_rows(*args) is None
    embed = _inputs(64, 16, torch.bfloat16)[0]
    assert token_rows(embed, ids, pos, cos, sin) is None              # a gradient may be wanted
    hook = embed.register_forward_hook(lambda *_: None)
    with torch.no_grad():
        assert token_rows(embed, ids, pos, cos, sin) is None
        hook.remove()
        assert token_rows(embed, ids, pos, cos, sin) is not None
