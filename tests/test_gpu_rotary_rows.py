"""The rotary operator's split of tokens over workgroups: many tokens a workgroup, one, several workgroups a token, and
the sizes around them."""
import pytest
import torch

from chunk_attn import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("neox", [True, False])
@pytest.mark.parametrize("tokens,heads,kv_heads,head_size", [
    (5000, 1, 0, 16), (301, 1, 1, 64), (77, 16, 15, 128), (9, 16, 16, 128), (7, 31, 2, 128), (3, 40, 25, 128), (1, 8, 8, 64)])
def test_every_row_is_turned_once(neox, tokens, heads, kv_heads, head_size):
    g = torch.Generator().manual_seed(tokens)
    q, k = (torch.randn(tokens, h * head_size, generator=g).half().cuda() for h in (heads, max(kv_heads, 1)))
    k_all = k if kv_heads else k[:, :0]
    angles = torch.rand(100, head_size // 2, generator=g) * 6.3
    table = torch.cat([angles.cos(), angles.sin()], dim=1).half().cuda()
    pos = torch.randint(0, 100, (tokens,), generator=g).cuda()
    cos, sin = (t[:, None] for t in table.double()[pos].chunk(2, dim=-1))
    want = []
    for x in (q, k):
        x = x.double().view(tokens, -1, head_size)
        a, b = (x.chunk(2, dim=-1) if neox else (x[..., 0::2], x[..., 1::2]))
        turned = (a * cos - b * sin, b * cos + a * sin)
        want.append((torch.cat(turned, dim=-1) if neox else torch.stack(turned, dim=-1).flatten(-2)).flatten(1))
    if kv_heads:
        capi.rotary_embedding(pos, q, k, head_size, table, neox)
    else:
        stream = torch.cuda.current_stream().cuda_stream
        capi._check(capi.load().ca_rotary_embedding(pos.data_ptr(), q.data_ptr(), None, table.data_ptr(), tokens, heads, 0,
                                                    head_size, head_size, 100, q.shape[1], 0, int(neox), stream))
    # fp32 products and sums of two terms, rounded to fp16 once
    for got, ref in ((q, want[0]), (k_all, want[1]))[:2 if kv_heads else 1]:
        assert ((got.double() - ref).abs() <= ref.abs() * 2.0 ** -11 + 2.0 ** -20).all()
