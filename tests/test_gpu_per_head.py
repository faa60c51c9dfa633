"""Streaming with a head per wave of whole sequences, against the tiles in turn and against fp64."""
import math

import pytest
import torch

from chunk_attn import capi

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _close(got, want):
    # each is rounded to fp16 once (half of 2^-10), the fp32 sums of some thousand weights differ by far less
    assert ((got.double() - want.double()).abs() <= want.double().abs() * 2.0 ** -10 + 2.0 ** -20).all()


@pytest.mark.parametrize("n,heads,c,lengths", [
    (32, 32, 64, [1023, 1024, 1000]),               # half a round of workgroups, a last chunk that is empty
    (64, 16, 32, [2047, 2080, 2049]),               # 64 chunks and more: their slots come in two loads
    (128, 8, 64, [4160, 4095, 4096, 4097]),
    (44, 24, 128, [1280, 1279, 1281, 1217])])
def test_whole_sequences_head_per_wave(n, heads, c, lengths):
    """Forwards and fused steps until last chunks have filled up and rolled over."""
    g = torch.Generator(device=DEV).manual_seed(n + c)
    own = [lengths[s % len(lengths)] for s in range(n)]
    mb = sum(m // c + 2 for m in own) * c * heads * 128 * 4 // (1 << 20) + 2
    attn = capi.Attention(heads, 128, c, memory_mb=mb, dtype=torch.float16, device=DEV)
    pairs, kept = [(0, 0), (n - 1, heads - 1), (n // 2, 3)], {}
    for s, m in enumerate(own):
        k, v = (torch.empty((m, heads, 128), dtype=torch.float16, device=DEV).normal_(generator=g) for _ in range(2))
        attn.add_seq([100_000 * (s + 1) + i for i in range(m)], k, v)
        for a, h in pairs:
            if a == s:
                kept[a, h] = [k[:, h].double(), v[:, h].double()]
    attn.refresh_kernel_context()
    assert attn.ctx.plan_info().stream_per_head == 1 and attn.ctx.plan_info().n_part_rows == 0

    def check(out, q):
        for (s, h), (k, v) in kept.items():
            p = torch.softmax((k * q[s, h].double()).sum(-1) / math.sqrt(128), dim=0)
            want = (p[:, None] * v).sum(0)
            assert ((out[s, h].double() - want).abs() <= want.abs() * 2.0 ** -11 + 2.0 ** -16).all()

    for step in range(8):
        q, k, v = (torch.empty((n, heads, 128), dtype=torch.float16, device=DEV).normal_(generator=g) for _ in range(3))
        out = attn.decode_step([50_000_000 + 1000 * step + s for s in range(n)], q, k, v)
        for (s, h), held in kept.items():
            held[0], held[1] = torch.cat([held[0], k[s, h].double()[None]]), torch.cat([held[1], v[s, h].double()[None]])
        check(out, q)
        attn.reserve()
        attn.refresh_kernel_context()
        assert attn.ctx.plan_info().stream_per_head == 1
        assert torch.equal(attn.forward(q), out)
    attn.ctx.set_plan(0, max(4, 256 // c))          # the tiles in turn
    attn.refresh_kernel_context(force=True)
    assert attn.ctx.plan_info().stream_per_head == 0
    _close(attn.forward(q), out)
    attn.ctx.set_plan(0, 0)
    attn.ctx.set_schedule(1)                        # one launch, whose workgroups wait for one another: not a wave's own head
    attn.refresh_kernel_context(force=True)
    assert attn.ctx.plan_info().stream_per_head == 0
    _close(attn.forward(q), out)
    attn.ctx.set_schedule(0)
    attn.refresh_kernel_context(force=True)
    assert torch.equal(attn.forward(q), out)
