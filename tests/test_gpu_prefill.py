"""Causal attention of whole prompts against fp64 on the CPU, at the sizes where the kernel's tiles end:
64-key tiles, in launches of more workgroups of 64 rows 32-key tiles, 16 rows per wave."""
import math

import pytest
import torch

from chunk_attn import capi

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def reference(q, k, v):
    q, k, v = (t.double().transpose(1, 2).contiguous() for t in (q, k, v))
    n = q.shape[2]
    scores = (q @ k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[3])
    future = torch.ones(n, n, dtype=torch.bool).triu(1)
    return (torch.softmax(scores.masked_fill(future, float("-inf")), dim=-1) @ v).transpose(1, 2)


@pytest.mark.parametrize("batch,n,heads", [
    (1, 1, 1), (2, 15, 3), (1, 16, 8), (3, 63, 2), (1, 64, 8), (2, 65, 5), (1, 127, 2), (1, 129, 8),
    (1, 192, 8), (2, 193, 1),
    (8, 130, 16), (16, 128, 16), (37, 33, 8), (2, 513, 32), (1, 1025, 32), (50, 31, 8), (3, 161, 45), (1, 800, 31)])
def test_causal_attention_at_tile_edges(batch, n, heads):
    g = torch.Generator().manual_seed(n * 100 + heads)
    # scores of a few units either way: the running maximum moves, and small probabilities matter
    q, k, v = (torch.randn(batch, n, heads, 128, generator=g).half() for _ in range(3))
    q *= 2
    out = capi.causal_attention(q.cuda(), k.cuda(), v.cuda()).cpu().double()
    want = reference(q, k, v)
    # the output's own rounding is 2^-11 of it at most; sums of n fp32 terms add less than 2^-16 of max |v| < 6
    assert ((out - want).abs() <= want.abs() * 2.0 ** -11 + 6 * 2.0 ** -16).all()


@pytest.mark.parametrize("batch,n,heads", [
    (37, 31, 16), (52, 64, 12), (26, 65, 12), (13, 97, 24), (20, 129, 10), (5, 193, 42), (13, 513, 8), (2, 600, 39), (1, 1633, 30),
    (1, 577, 64), (9, 64, 64), (3, 601, 25)])
def test_causal_attention_of_many_workgroups(batch, n, heads):
    """32-key tiles: from 577 workgroups on, from 769 for prompts of 600 tokens and more (the last two lie before
    the lines)."""
    test_causal_attention_at_tile_edges(batch, n, heads)


def test_what_a_row_must_not_see_and_extreme_scores():
    """Tokens after a row change nothing in it; scores of +-3e4 neither overflow nor lose the row."""
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(1, 200, 8, 128, generator=g).half() for _ in range(3))
    q[:, 50:] *= 60
    k[:, 50:] *= 60
    whole = capi.causal_attention(q.cuda(), k.cuda(), v.cuda()).cpu()
    assert torch.isfinite(whole).all()
    first = capi.causal_attention(*(t[:, :70].contiguous().cuda() for t in (q, k, v))).cpu()
    assert torch.equal(whole[:, :70], first)
    want = reference(q, k, v)
    # scores of |s| <= 3e4 carry an fp32 rounding of 2^-24 |s| sqrt(128): at most 2^-6 of a probability
    assert ((whole.double() - want).abs() <= want.abs() * 2.0 ** -6 + 6 * 2.0 ** -6).all()
    assert torch.equal(whole[:, :50], capi.causal_attention(*(t[:, :50].contiguous().cuda() for t in (q, k, v))).cpu())


def test_refused_inputs():
    q = torch.zeros(1, 8, 2, 128, dtype=torch.float16, device="cuda")
    for bad in (q.float(), q[:, ::2], torch.zeros(1, 8, 2, 64, dtype=torch.float16, device="cuda"), q.cpu(),
                torch.zeros(8 * 256 + 1, dtype=torch.float16, device="cuda")[1:].view(1, 8, 2, 128)):
        assert not capi.causal_attention_takes(bad, bad, bad)
        with pytest.raises(RuntimeError):
            capi.causal_attention(bad, bad, bad)
    assert not capi.causal_attention_takes(q, q, torch.zeros_like(q, requires_grad=True))


@pytest.mark.parametrize("batch,n,heads", [(1, 200, 8), (8, 300, 16)])       # 64-key tiles, 32-key tiles
def test_later_rows_of_a_wave_change_nothing_in_earlier_ones(batch, n, heads):
    """Ordinary scores, whose running maxima move by less than the kernel's slack, beside rows of the same 16
    whose maxima jump."""
    g = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(batch, n, heads, 128, generator=g).half().cuda() for _ in range(3))
    first = capi.causal_attention(q, k, v)
    q[:, 150:] *= 8                                                       # rows 150 .. 159 share a wave with 144 .. 149
    second = capi.causal_attention(q, k, v)
    assert torch.equal(first[:, :150], second[:, :150]) and not torch.equal(first[:, 150:], second[:, 150:])


@pytest.mark.parametrize("batch,n,heads", [(1, 200, 8), (8, 300, 16)])       # 64-key tiles, 32-key tiles
def test_infinite_and_undefined_scores(batch, n, heads):
    """A key of minus infinity is not attended, one of infinity or NaN spoils the rows that see it; rows before stay
    as they were."""
    g = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(batch, n, heads, 128, generator=g).half() for _ in range(3))
    q[..., 0] = 1
    inf = float("inf")
    k[0, 100, 1, 0], k[0, 120, 2, 0], k[0, 130, 3, 5], k[0, 0, 4, 0], k[0, 63:66, 5, 0] = -inf, inf, float("nan"), -inf, -inf
    out = capi.causal_attention(q.cuda(), k.cuda(), v.cuda()).cpu().double()
    want = reference(q, k, v)
    assert torch.equal(torch.isnan(out), torch.isnan(want))
    assert torch.isnan(want).any(-1).sum() == (n - 120) + (n - 130) + 1
    ok = ~torch.isnan(want)
    assert ((out - want).abs() <= want.abs() * 2.0 ** -11 + 6 * 2.0 ** -16)[ok].all()


@pytest.mark.parametrize("batch,n,heads,chunk,same", [
    (1, 1, 1, 32, 0), (1, 63, 3, 64, 0), (2, 64, 8, 64, 0), (3, 65, 2, 32, 40), (2, 256, 8, 64, 256), (8, 130, 2, 32, 64),
    (1, 2048, 2, 32, 0), (2, 1061, 1, 32, 700), (3, 300, 5, 128, 150)])
def test_attention_and_insertion_in_one_launch(batch, n, heads, chunk, same):
    """Prompts that share `same` tokens, with up to 64 chunks and more, into a cache that holds one already: output,
    indices, tree and every row of the pools as from the separate calls."""
    g = torch.Generator(device=DEV).manual_seed(batch * n + heads)
    q, k, v = (torch.empty((batch, n, heads, 128), dtype=torch.float16, device=DEV).normal_(generator=g) for _ in range(3))
    first = torch.empty((chunk + 3, heads, 128), dtype=torch.float16, device=DEV).normal_(generator=g)
    prompts = [list(range(min(same, n))) + [1000 * (s + 1) + t for t in range(n - same)] for s in range(batch)]
    found = []
    for joined in (True, False):
        cache = capi.Attention(heads, 128, chunk, memory_mb=64, dtype=torch.float16, device=torch.device(DEV))
        for pool in cache.pool_views():
            pool.zero_()
        cache.add_seq(list(range(chunk + 3)), first, first)
        if joined:
            out, index = cache._prefill_attention(prompts, q, k, v)
        else:
            out, index = capi.causal_attention(q, k, v), [cache.add_seq(p, k[i], v[i]) for i, p in enumerate(prompts)]
        assert not cache.ctx.valid
        found.append((out, index, cache.tree.get_chunks(), cache.pool_views(), cache))
    a, b = found
    assert torch.equal(a[0], b[0]) and a[1] == b[1] and (a[2] == b[2]).all()
    assert all(torch.equal(x, y) for x, y in zip(a[3], b[3]))


def test_a_prompt_the_cache_cannot_take_leaves_those_before_it_with_their_rows():
    k = torch.randn((2, 400, 16, 128), device=DEV).half()
    cache = capi.Attention(16, 128, 64, memory_mb=4, dtype=torch.float16, device=torch.device(DEV))   # 8 chunks
    for pool in cache.pool_views():
        pool.zero_()
    with pytest.raises(RuntimeError):
        cache._prefill_attention([list(range(400)), list(range(1000, 1400))], k, k, k)
    rows = [(slot, m) for slot, m, begin, _ in cache.tree.get_chunks() if begin == 0]
    assert sum(m for _, m in rows) == 400
    for pool in cache.pool_views():
        assert torch.equal(torch.cat([pool[slot][:, :m] for slot, m in rows[:7]], dim=1).transpose(0, 1), k[0])


def test_prompts_that_are_not_the_caches_are_left_to_the_separate_calls():
    q = torch.zeros((1, 40, 2, 128), device=DEV).half()
    cache = capi.Attention(2, 128, 64, memory_mb=2, dtype=torch.float16, device=torch.device(DEV))
    for prompts in ([], [list(range(39))], [tuple(range(40))], [[1 << 40] * 40], [[0.5] * 40], [list(range(40))] * 2):
        assert cache._prefill_attention(prompts, q, q, q) is None
    assert cache._prefill_attention([list(range(40))], *[q[:, :, :1].contiguous()] * 3) is None
    assert cache.tree.n_seqs == 0


@pytest.mark.parametrize("chunk", [48, 20])
def test_prefill_into_chunks_of_a_size_that_no_decode_attention_takes(chunk):
    """Such a cache is filled like any other, by the attention's own launch, by the layer and by the small model; only a
    decode forward over it is refused."""
    from chunk_attn.llama_layer import LlamaChunkAttention
    from chunk_attn.models.sequence import Sequence
    from chunk_attn.models.tiny_lm import AttentionOnlyLM
    test_attention_and_insertion_in_one_launch(2, 3 * chunk + 7, 2, chunk, chunk + 3)
    prompts = [[100 * s + t for t in range(2 * chunk + 5)] for s in range(2)]
    layer = LlamaChunkAttention(256, 2, max_position_embeddings=256)
    x = torch.randn((2, 2 * chunk + 5, 256), device=DEV).half()
    positions = torch.arange(2 * chunk + 5, device=DEV).expand(2, -1).contiguous()
    with torch.inference_mode():
        outs, rows = [], []
        for size in (chunk, 64):
            cache = capi.Attention(2, 128, size, memory_mb=8, dtype=torch.float16, device=torch.device(DEV))
            outs.append(layer(x, prompts, positions, cache, True))
            assert layer.last_indices == [0, 1]
            rows.append([torch.cat([pool[slot][:, :m] for slot, m, b, e in cache.get_chunks() if b <= s < e], dim=1)
                         for s in range(2) for pool in cache.pool_views()])
            if size == chunk:
                with pytest.raises(RuntimeError, match="unsupported chunk_size"):
                    cache.forward(torch.zeros((2, 2, 128), device=DEV).half())
        assert torch.equal(*outs) and all(torch.equal(a, b) for a, b in zip(*rows))
        logits = []
        for size, hooked in ((chunk, False), (chunk, True), (64, False)):
            model = AttentionOnlyLM(60, 256, 2, 2, chunk_size=size, memory_mb=8, seed=7)
            if hooked:                                       # the modules' own calls
                model.norm.register_forward_hook(lambda m, a, out: None)
            logits.append(model.logits([Sequence(list(range(50)))], model.create_kv_caches(), True))
        assert torch.equal(logits[0], logits[1]) and torch.equal(logits[0], logits[2])


@pytest.mark.parametrize("tree_chunk,tree_chunks,match", [
    (128, 16, "as many tokens"), (32, 16, "as many tokens"), (64, 16, "outside the pool")])
def test_a_tree_whose_chunks_are_not_the_contexts(tree_chunk, tree_chunks, match):
    """Larger chunks, smaller ones, more of them than the pool has: the prompt that shows it is refused and not in the
    tree; those before it stay, with their rows."""
    import ctypes
    n, fits = 100 if tree_chunk > 64 else 64, tree_chunk == 64
    k = torch.randn((4, n, 2, 128), device=DEV).half()
    cache = capi.Attention(2, 128, 64, memory_mb=1, dtype=torch.float16, device=torch.device(DEV))
    pool_chunks = 4                                          # of the pool, for the context: two prompts and their tails
    ctx = capi.KernelContext(2, 128, 64, cache.key_storage.data_ptr(), cache.value_storage.data_ptr(), pool_chunks)
    tree = capi.Tree(tree_chunk, tree_chunks)
    for pool in cache.pool_views():
        pool.zero_()
    prompts = [1000 * s + t for s in range(4) for t in range(n)]
    out, index = torch.empty_like(k), (ctypes.c_int32 * 4)(*[7] * 4)
    with pytest.raises(RuntimeError, match=match):
        capi._launch(k.device, ctx._lib.ca_prefill_attention, ctx._h, tree._h, (ctypes.c_int32 * len(prompts))(*prompts), 4, n,
                     k.data_ptr(), k.data_ptr(), k.data_ptr(), out.data_ptr(), index)
    taken = 2 if fits else 0
    assert tree.n_seqs == taken and list(index) == list(range(taken)) + [-1] + [7] * (3 - taken)
    rows = tree.get_chunks()
    for s in range(taken):
        (slot,) = [slot for slot, m, b, _ in rows if b == s and m > 0]
        for pool in cache.pool_views():
            assert torch.equal(pool[slot].transpose(0, 1), k[s])
    assert all(not pool[slot].any() for pool in cache.pool_views() for slot in range(cache.max_chunks)
               if slot not in [r[0] for r in rows])
    assert torch.equal(out, capi.causal_attention(k, k, k))
