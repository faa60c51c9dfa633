"""The projection kernel against fp64 at the edges of its tiles: 16, 32 and 64 rows, columns past the last whole
tile, one to many units of 64 elements for each of the eight waves."""
import pytest
import torch

from chunk_attn import capi
from chunk_attn.llama_layer import LlamaChunkAttention

pytestmark = pytest.mark.gpu


def _draw(g, *shape, sigma=1.0):
    return (torch.randn(*shape, generator=g) * sigma).half().cuda()


def _close(got, want, n_in):
    # one rounding to fp16 (2^-11 of the value), and n_in fp32 products of unit variance summed in any order:
    # at most 2^-24 * n_in of their absolute sum, which is below n_in * n_in ** -0.5
    assert got.shape == want.shape
    assert ((got.double() - want).abs() <= want.abs() * 2.0 ** -11 + n_in ** 1.5 * 2.0 ** -24 + 2.0 ** -20).all()


@pytest.mark.parametrize("rows,n_out,n_in", [
    (1, 1, 64), (1, 17, 128), (3, 500, 256), (8, 8000, 1024), (15, 128, 448), (16, 130, 512), (16, 64, 1088),
    (16, 48, 1536), (9, 40, 4096), (17, 33, 64), (32, 96, 576), (33, 31, 1024), (64, 512, 256), (65, 130, 320),
    (252, 1024, 1024), (100, 4100, 1024), (129, 8192, 192), (2048, 512, 512)])
def test_linear_at_tile_edges(rows, n_out, n_in):
    g = torch.Generator().manual_seed(rows * 7 + n_out)
    x, w = _draw(g, rows, n_in), _draw(g, n_out, n_in, sigma=n_in ** -0.5)
    layer = torch.nn.Linear(n_in, n_out, bias=False, dtype=torch.float16, device="cuda")
    with torch.no_grad():
        layer.weight.copy_(w)
        assert capi.projection_takes(x, layer)
    guard = torch.full((rows * n_out + 64,), 3.0, dtype=torch.float16, device="cuda")
    out = guard[:rows * n_out].view(rows, n_out)
    capi._check(capi.load().ca_linear(x.data_ptr(), w.data_ptr(), out.data_ptr(), rows, n_out, n_in,
                                      torch.cuda.current_stream().cuda_stream))
    _close(out, x.double() @ w.double().t(), n_in)
    assert (guard[rows * n_out:] == 3.0).all()
    assert torch.equal(capi.linear(x, w), out)


@pytest.mark.parametrize("rows,heads,n_in", [(1, 1, 128), (5, 3, 384), (16, 8, 1024), (8, 12, 1536), (17, 2, 256),
                                             (63, 3, 1024), (252, 8, 1024), (130, 32, 4096), (700, 12, 1472)])
def test_qkv_rotary(rows, heads, n_in):
    g = torch.Generator().manual_seed(rows + heads)
    x = _draw(g, rows, n_in)
    ws = [_draw(g, heads * 128, n_in, sigma=n_in ** -0.5) for _ in range(3)]
    angles = torch.rand(300, 64, generator=g) * 6.3
    table = torch.cat([angles.cos(), angles.sin()], dim=1).half().cuda()
    positions = torch.randint(-3, 303, (rows,), generator=g)           # outside the table: clamped into it
    q, k, v = capi.qkv_rotary(x, *ws, positions.cuda(), table)
    cos, sin = table.double()[positions.clamp(0, 299).cuda()].chunk(2, dim=-1)
    for got, w, turned in ((q, ws[0], True), (k, ws[1], True), (v, ws[2], False)):
        want = (x.double() @ w.double().t()).view(rows, heads, 128)
        if turned:
            a, b = want.chunk(2, dim=-1)
            want = torch.cat([a * cos[:, None] - b * sin[:, None], b * cos[:, None] + a * sin[:, None]], dim=-1)
        _close(got, want.reshape(rows, -1), 2 * n_in)


@pytest.mark.parametrize("batch,heads,chunk", [(1, 2, 32), (9, 8, 64), (17, 2, 128)])
def test_layer_decode_writes_the_pool_as_the_library_path_does(batch, heads, chunk):
    """The folded step and the one with torch projections leave the same cache (but for fp16 roundings), over
    steps in which last chunks fill up, and refuse the same calls."""
    hidden, n = heads * 128, chunk - 2
    outs, caches = [], []
    for folded in (True, False):
        g = torch.Generator().manual_seed(batch)
        layer = LlamaChunkAttention(hidden, heads, device="cuda")
        with torch.no_grad():
            for p in (layer.q_proj, layer.k_proj, layer.v_proj, layer.o_proj):
                p.weight.copy_(_draw(g, hidden, hidden, sigma=hidden ** -0.5))
        if not folded:
            for p in (layer.q_proj, layer.o_proj):
                p.register_forward_hook(lambda module, args, out: out)   # something hangs on the module
        kv = capi.Attention(heads, 128, chunk, memory_mb=64, dtype=torch.float16, device=torch.device("cuda:0"))
        seqs = [[100 * s + t for t in range(n)] for s in range(batch)]
        out = []
        with torch.inference_mode():
            pos = torch.arange(n).repeat(batch, 1).cuda()
            out.append(layer(_draw(g, batch, n, hidden), seqs, pos, kv, True))
            for t in range(4):
                seqs = [s + [7] for s in seqs]
                out.append(layer(_draw(g, batch, 1, hidden), seqs, torch.full((batch, 1), n + t).cuda(), kv, False))
            with pytest.raises(RuntimeError, match="num of seqs"):
                layer(_draw(g, batch + 1, 1, hidden), seqs + [[1]], torch.zeros(batch + 1, 1, dtype=torch.int64).cuda(), kv, False)
        outs.append(out)
        caches.append((kv.tree.get_chunks(), [p.float() for p in kv.pool_views()]))
    assert (caches[0][0] == caches[1][0]).all()
    for a, b in zip(*outs):
        assert (a.float() - b.float()).norm() <= 4e-3 * b.float().norm()
    for slot, n_tokens, _, _ in caches[0][0]:
        for a, b in zip(caches[0][1], caches[1][1]):
            a, b = a[slot][:, :n_tokens], b[slot][:, :n_tokens]
            # the library path rounds the projection, then the rotation: two roundings of 2^-11 against one
            assert ((a - b).abs() <= 2.0 ** -9 * b.abs().amax()).all()


def test_layer_takes_the_pybind_cache_too():
    from chunk_attn import Attention
    outs = []
    for cls in (capi.Attention, Attention):
        g = torch.Generator().manual_seed(3)
        layer = LlamaChunkAttention(256, 2, device="cuda")
        kv = cls(2, 128, 64, memory_mb=16, dtype=torch.float16, device=torch.device("cuda:0"))
        with torch.inference_mode():
            pos = torch.arange(20).repeat(3, 1).cuda()
            x, y = _draw(g, 3, 20, 256), _draw(g, 3, 1, 256)
            for p, w in zip((layer.q_proj, layer.k_proj, layer.v_proj, layer.o_proj), (_draw(g, 256, 256, sigma=0.06) for _ in range(4))):
                p.weight.copy_(w)
            layer(x, [[s] * 20 for s in range(3)], pos, kv, True)
            outs.append(layer(y, [[s] * 21 for s in range(3)], torch.full((3, 1), 20).cuda(), kv, False).float())
    assert (outs[0] - outs[1]).norm() <= 4e-3 * outs[1].norm()


def test_model_with_its_adds_in_the_norms():
    """A hook on a norm keeps the adds on their own: the same logits but for the roundings of the residual."""
    from chunk_attn.models.sequence import Sequence
    from chunk_attn.models.tiny_lm import AttentionOnlyLM
    runs = []
    for hooked in (False, True):
        model = AttentionOnlyLM(300, 256, 2, 3, chunk_size=32, memory_mb=16, seed=4)
        seen = []
        if hooked:
            model.input_norms[1].register_forward_hook(lambda m, a, out: seen.append(out.clone()))
        caches, out = model.create_kv_caches(), []
        with torch.inference_mode():
            seqs = [Sequence([5 * s + t for t in range(40)]) for s in range(3)]
            out.append(model.logits(seqs, caches, True))
            seqs.sort(key=lambda s: s.index)
            for t in range(3):
                for s in seqs:
                    s.append(7 + t)
                out.append(model.logits(seqs, caches, False))
        assert len(seen) == (4 if hooked else 0)
        runs.append(out)
    for a, b in zip(*runs):
        # each norm's input differs by one fp16 rounding (2^-11) of the residual at most
        assert (a.float() - b.float()).norm() <= 4e-3 * b.float().norm()
    assert AttentionOnlyLM(50, 128, 1, 0, memory_mb=1).logits([Sequence([1, 2])], [], True).shape == (1, 50)


def test_what_the_projection_leaves_to_torch():
    x = torch.zeros(4, 256, dtype=torch.float16, device="cuda")
    lin = torch.nn.Linear(256, 128, bias=False, dtype=torch.float16, device="cuda")
    assert not capi.projection_takes(x, lin)                            # a gradient is wanted
    with torch.no_grad():
        assert capi.projection_takes(x, lin)
        assert not capi.projection_takes(x.float(), lin)
        assert not capi.projection_takes(torch.zeros(4, 512, dtype=torch.float16, device="cuda")[:, ::2], lin)
        assert not capi.projection_takes(torch.zeros(8192, 256, dtype=torch.float16, device="cuda"), lin)
        assert not capi.projection_takes(x, torch.nn.Linear(256, 128, dtype=torch.float16, device="cuda"))
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert not capi.projection_takes(x, lin)
        handle = lin.register_forward_hook(lambda *a: None)
        assert not capi.projection_takes(x, lin)
        handle.remove()
        assert capi.projection_takes(x, lin)


def test_model_keeps_what_a_hook_on_an_output_projection_holds():
    """The tensor a hook keeps is the projection's output still, not the sum or norm that followed it."""
    from chunk_attn.models.sequence import Sequence
    from chunk_attn.models.tiny_lm import AttentionOnlyLM
    model = AttentionOnlyLM(300, 256, 2, 2, chunk_size=32, memory_mb=16, seed=5)
    kept, copies = [], []
    model.layers[0].o_proj.register_forward_hook(lambda m, a, out: (kept.append(out), copies.append(out.clone())) and None)
    with torch.inference_mode():
        model.logits([Sequence(list(range(40)))], model.create_kv_caches(), True)
    assert len(kept) == 1 and (kept[0] == copies[0]).all()


def test_causal_attention_leaves_forward_mode_to_torch():
    from torch.autograd import forward_ad
    q = torch.zeros(1, 8, 2, 128, dtype=torch.float16, device="cuda")
    assert capi.causal_attention_takes(q, q, q)
    with forward_ad.dual_level():
        assert not capi.causal_attention_takes(q, q, q)
    assert capi.causal_attention_takes(q, q, q)


def test_model_with_its_adds_in_the_norms_keeps_every_bit():
    from chunk_attn.models.sequence import Sequence
    from chunk_attn.models.tiny_lm import AttentionOnlyLM
    out = []
    for hooked in (False, True):
        model = AttentionOnlyLM(300, 1024, 8, 3, chunk_size=32, memory_mb=16, seed=4)
        if hooked:
            model.input_norms[1].register_forward_hook(lambda m, a, out: None)
        caches = model.create_kv_caches()
        with torch.inference_mode():
            seq = Sequence(list(range(200)))
            out.append([model.logits([seq], caches, True)])
            seq.append(7)
            out[-1].append(model.logits([seq], caches, False))
    assert all(torch.equal(a, b) for a, b in zip(*out))


def test_projections_refuse_what_their_kernels_cannot_read():
    """Fewer columns, other types, strides, alignments and devices: refused before anything is launched or kept."""
    heads, n_in, n = 2, 256, 3
    x = torch.zeros(n, n_in, dtype=torch.float16, device="cuda")
    w = torch.zeros(n_in, n_in, dtype=torch.float16, device="cuda")
    flat = torch.zeros(n_in * n_in + 1, dtype=torch.float16, device="cuda")
    bad_x = [x.float(), x.cpu(), x.t().contiguous().t(), flat[1:1 + n * n_in].view(n, n_in), x[:, :100].contiguous(), x[:, :0]]
    bad_w = [w[:, :128].contiguous(), w.float(), w.bfloat16(), torch.empty(n_in, n_in, dtype=torch.float16, device="cuda").t(),
             w.cpu(), flat[1:].view(n_in, n_in), w.view(-1)]
    table = torch.zeros(64, 128, dtype=torch.float16, device="cuda")
    pos = torch.zeros(n, dtype=torch.int64, device="cuda")
    kv = capi.Attention(heads, 128, 32, memory_mb=4, dtype=torch.float16, device=torch.device("cuda:0"))
    for s in range(n):
        kv.add_seq([s] * 5, *(torch.zeros(5, heads, 128, dtype=torch.float16, device="cuda") for _ in range(2)))
    kv.refresh_kernel_context()
    calls = [(lambda a, b: capi.linear(a, b), 1), (lambda a, *b: capi.qkv_rotary(a, *b, pos, table), 3),
             (lambda a, *b: kv.project_append_rotary([7] * n, a, *b, table, pos), 3),
             (lambda a, *b: kv.layer_decode([7] * n, a, *b, table, pos), 4)]
    before = kv.tree.dump()
    for call, count in calls:
        cases = [(bad, *[w] * count) for bad in bad_x]
        cases += [(x, *[w] * at, bad, *[w] * (count - at - 1)) for bad in bad_w for at in range(count)]
        for case in cases:
            with pytest.raises(RuntimeError):
                call(*case)
    assert kv.tree.dump() == before and kv.ctx.delta_tokens == 0
    for call, count in calls:
        call(x, *[w] * count)


def test_a_refused_decode_pass_leaves_the_cache_as_it_was():
    """Every argument of ca_layer_decode is looked at before the tree, the pool and the tables move on."""
    import ctypes
    heads, n = 2, 3
    t = lambda *shape: torch.ones(shape, dtype=torch.float16, device="cuda")
    x, w, q, y, table = t(n, 256), t(256 * 256 + 8) / 256, t(2, n, 256), t(n, 256), t(64, 128)   # products of 1
    pos = torch.zeros(n, dtype=torch.int64, device="cuda")
    tokens = (ctypes.c_int32 * n)(7, 7, 7)

    def cache(chunk):
        kv = capi.Attention(heads, 128, chunk, memory_mb=4, dtype=torch.float16, device=torch.device("cuda:0"))
        for s in range(n):
            kv.add_seq([s] * chunk, t(chunk, heads, 128), t(chunk, heads, 128))   # full: a pass needs new last chunks
        return kv

    def args(**changed):
        a = dict(x=x.data_ptr(), n_in=256, wq=w.data_ptr(), wk=w.data_ptr(), wv=w.data_ptr(), wo=w.data_ptr(), n_out=256,
                 positions=pos.data_ptr(), table=table.data_ptr(), max_position=64, q=q[0].data_ptr(), attn=q[1].data_ptr(), y=y.data_ptr())
        assert set(changed) <= set(a)
        return list(dict(a, **changed).values())

    def call(kv, a):
        return kv.ctx._lib.ca_layer_decode(kv.ctx._h, kv.tree._h, tokens, n, *a, torch.cuda.current_stream().cuda_stream)

    bad = [{k: 0} for k in ("x", "wq", "wk", "wv", "wo", "n_in", "n_out", "positions", "table", "max_position", "q", "attn", "y")]
    bad += [{"n_in": 100}, {"n_out": -5}, {"wo": w.data_ptr() + 2}, {"attn": q[1].data_ptr() + 2}, {"wq": w.data_ptr() + 4},
            {"q": q.data_ptr() + 2}, {"table": table.data_ptr() + 2}]
    for kv, changes in ((cache(32), bad), (cache(48), [{}])):               # chunks of 48: no attention kernel
        before, pools = kv.tree.dump(), [p.clone() for p in kv.pool_views()]
        for change in changes:
            assert call(kv, args(**change)) < 0, change
        assert kv.tree.dump() == before and kv.ctx.delta_tokens == 0
        assert all(torch.equal(a, b) for a, b in zip(pools, kv.pool_views()))
    kv = cache(32)
    assert call(kv, args()) == 0 and kv.tree.n_seqs == n and torch.isfinite(y).all()


def test_output_of_another_cache_is_not_taken_for_granted():
    """A cache of another class may return another type: torch's product refuses it, the kernel must not read it."""
    class Wide(capi.Attention):
        def forward(self, q, partition=0):
            return super().forward(q, partition).float()

    layer = LlamaChunkAttention(256, 2, device="cuda")
    kv = Wide(2, 128, 64, memory_mb=16, dtype=torch.float16, device=torch.device("cuda:0"))
    with torch.inference_mode():
        layer(_draw(torch.Generator().manual_seed(1), 1, 5, 256), [[1] * 5], torch.arange(5)[None].cuda(), kv, True)
        with pytest.raises(RuntimeError):
            layer(torch.zeros(1, 1, 256, dtype=torch.float16, device="cuda"), [[1] * 6], torch.full((1, 1), 5).cuda(), kv, False)


def test_gradient_of_another_cache_goes_through_the_output_projection():
    """A cache of another class may return something learned: with frozen weights its gradient is the product's."""
    class Learned(capi.Attention):
        def forward(self, q, partition=0):
            return super().forward(q, partition) + self.offset

    layer = LlamaChunkAttention(256, 2, device="cuda").requires_grad_(False)
    kv = Learned(2, 128, 64, memory_mb=16, dtype=torch.float16, device=torch.device("cuda:0"))
    kv.offset = torch.zeros(1, 2, 128, dtype=torch.float16, device="cuda", requires_grad=True)
    layer(_draw(torch.Generator().manual_seed(1), 1, 5, 256), [[1] * 5], torch.arange(5)[None].cuda(), kv, True)
    out = layer(_draw(torch.Generator().manual_seed(2), 1, 1, 256), [[1] * 6], torch.full((1, 1), 5).cuda(), kv, False)
    out.sum().backward()
    want = layer.o_proj.weight.double().sum(0)
    # sums of 256 products with one in fp32, rounded to fp16
    assert ((kv.offset.grad.double().view(-1) - want).abs() <= want.abs() * 2.0 ** -11 + 2.0 ** -14).all()


@pytest.mark.parametrize("batch,heads,chunk", [(1, 2, 32), (9, 8, 64)])
def test_folded_projections_with_the_output_projection_on_its_own(batch, heads, chunk):
    """A hook on the output projection alone: q, k and v still come from one launch with their append, in steps of
    their own.  The cache is the whole pass's bit for bit, last chunks that fill up on the way included."""
    hidden, n = heads * 128, chunk - 2
    outs, caches, seen = [], [], []
    for hooked in (False, True):
        g = torch.Generator().manual_seed(batch)
        layer = LlamaChunkAttention(hidden, heads, device="cuda")
        with torch.no_grad():
            for p in (layer.q_proj, layer.k_proj, layer.v_proj, layer.o_proj):
                p.weight.copy_(_draw(g, hidden, hidden, sigma=hidden ** -0.5))
        if hooked:
            layer.o_proj.register_forward_hook(lambda module, args, out: seen.append(out))
        kv = capi.Attention(heads, 128, chunk, memory_mb=64, dtype=torch.float16, device=torch.device("cuda:0"))
        seqs = [[100 * s + t for t in range(n)] for s in range(batch)]
        with torch.inference_mode():
            out = [layer(_draw(g, batch, n, hidden), seqs, torch.arange(n).repeat(batch, 1).cuda(), kv, True)]
            for t in range(5):
                seqs = [s + [7] for s in seqs]
                out.append(layer(_draw(g, batch, 1, hidden), seqs, torch.full((batch, 1), n + t).cuda(), kv, False))
        outs.append(out)
        caches.append((kv.tree.dump(), kv.tree.get_chunks(), kv.pool_views()))
    assert len(seen) == 6 and caches[0][0] == caches[1][0]
    for slot, n_tokens, _, _ in caches[0][1]:
        assert all(torch.equal(a[slot][:, :n_tokens], b[slot][:, :n_tokens]) for a, b in zip(caches[0][2], caches[1][2]))
    for a, b in zip(*outs):
        # the two output projections sum in different orders and round once: a few units of 2^-11 at most
        assert (a.float() - b.float()).norm() <= 2e-3 * b.float().norm()


def test_infinities_and_nans_stay_in_their_rows():
    g = torch.Generator().manual_seed(2)
    x, w = _draw(g, 20, 256), _draw(g, 70, 256, sigma=0.06)
    x[3, 10], x[5, 200], x[19, 0] = float("inf"), float("nan"), float("-inf")
    x[7] = 60000.0
    want = (x.double() @ w.double().t())
    got = capi.linear(x, w).double()
    finite = want.abs() < 65504
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and (got[want > 65520] == float("inf")).all() and (got[want < -65520] == float("-inf")).all()
    assert ((got - want).abs() <= want.abs() * 2.0 ** -11 + 60000 * 256 ** 1.5 * 2.0 ** -24)[finite].all()


def test_launches_follow_the_current_stream():
    """The rows are written on a side stream behind a long wait: a launch anywhere else would read the old ones."""
    side = torch.cuda.Stream()
    g = torch.Generator().manual_seed(6)
    layer = LlamaChunkAttention(256, 2, device="cuda")
    x, y = _draw(g, 2, 30, 256), _draw(g, 2, 1, 256)
    pos, last = torch.arange(30).repeat(2, 1).cuda(), torch.full((2, 1), 30).cuda()
    outs = []
    for stream in (torch.cuda.current_stream(), side):
        kv = capi.Attention(2, 128, 64, memory_mb=16, dtype=torch.float16, device=torch.device("cuda:0"))
        a, b = torch.zeros_like(x), torch.zeros_like(y)
        torch.cuda.synchronize()
        with torch.inference_mode(), torch.cuda.stream(stream):
            torch.cuda._sleep(20_000_000)
            a.copy_(x)
            b.copy_(y)
            outs.append([layer(a, [[s] * 30 for s in range(2)], pos, kv, True), layer(b, [[s] * 31 for s in range(2)], last, kv, False),
                         capi.linear(b, layer.o_proj.weight)])
        torch.cuda.synchronize()
    assert all(torch.equal(s, t) and t.abs().max() > 0 for s, t in zip(*outs))
