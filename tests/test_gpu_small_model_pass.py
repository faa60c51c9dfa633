"""The small model's native pass against its modules' own calls."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,layers,prompts,chunk,vocab", [
    (128, 1, [1, 5], 32, 40), (1024, 3, [449, 30, 449], 64, 300), (512, 2, [900, 65, 64, 63], 128, 1001),
    # residuals in the output projection's tiles of 128 x 128 and 64 x 128, and of 128 x 256; more new chunks than one
    # launch copies
    (1024, 1, [3001, 1100], 32, 60), (1536, 2, [660, 2000], 64, 60), (2048, 1, [2100], 64, 60)])
def test_native_model_pass_keeps_every_bit(hidden, layers, prompts, chunk, vocab):
    """One native call a pass against the modules' own calls (a hook on a norm keeps them): prompts on both sides of
    the ids that one launch takes, decode steps over which last chunks fill up, the caches afterwards."""
    from chunk_attn.models.sequence import Sequence
    from chunk_attn.models.tiny_lm import AttentionOnlyLM
    runs = []
    for hooked in (False, True):
        model = AttentionOnlyLM(vocab, hidden, hidden // 128, layers, chunk_size=chunk, memory_mb=32, seed=6)
        if hooked:
            model.norm.register_forward_hook(lambda m, a, out: None)
        caches, running, out = model.create_kv_caches(), [], []
        with torch.inference_mode():
            for p in prompts:
                seq = Sequence([t * 7 % vocab for t in range(p)])
                assert hooked or model._plain_pass([seq], [seq.tokens], caches, True, torch.device("cuda:0")) is not None
                out.append(model.logits([seq], caches, True))
                running.insert(seq.index, seq)
                assert all(layer.last_indices == [seq.index] for layer in model.layers)
            for t in range(5):
                for s, seq in enumerate(running):
                    seq.append((11 * t + 3 * s) % vocab)
                out.append(model.logits(running, caches, False))
            if not hooked:
                before = [c.tree.get_chunks() for c in caches]
                for bad in (vocab, -1):
                    with pytest.raises(RuntimeError, match="vocabulary"):
                        model.logits([Sequence([0, bad])], caches, True)
                assert all((a == c.tree.get_chunks()).all() for a, c in zip(before, caches))
        rows = [c.tree.get_chunks() for c in caches]
        pools = [[p[slot][:, :n].clone() for slot, n, _, _ in r for p in c.pool_views()] for r, c in zip(rows, caches)]
        runs.append((out, rows, pools))
    assert all(torch.equal(a, b) for a, b in zip(runs[0][0], runs[1][0]))
    for a, b in zip(*(r[1] for r in runs)):
        assert (a == b).all()
    for a, b in zip(*(r[2] for r in runs)):
        assert all(torch.equal(x, y) for x, y in zip(a, b))


def test_what_the_native_pass_leaves_to_the_modules(monkeypatch):
    from chunk_attn import capi
    from chunk_attn.models.sequence import Sequence
    from chunk_attn.models.tiny_lm import AttentionOnlyLM
    dev = torch.device("cuda:0")
    model = AttentionOnlyLM(60, 256, 2, 2, chunk_size=32, memory_mb=8, seed=7)
    caches = model.create_kv_caches()
    ids = list(range(40))

    def taken(prefill=True, seqs=1, tokens=ids, kv=caches):
        with torch.inference_mode():
            return model._plain_pass([None] * seqs, [tokens] * seqs, kv, prefill, dev) is not None

    assert taken() and taken(prefill=False, tokens=[3]) and taken(prefill=False, seqs=5, tokens=[3])
    assert not taken(seqs=2) and not taken(tokens=[]) and not taken(seqs=0)       # several prompts, none
    assert not taken(tokens=[2 ** 40]) and not taken(tokens=["a"])                # ids that are no 32-bit numbers
    assert not taken(kv=caches[:1]) and not taken(kv=[caches[0], object()])
    assert not taken(kv=[caches[0], capi.Attention(3, 128, 32, memory_mb=8, dtype=torch.float16, device=dev)])
    assert not taken(tokens=[1] * 40000)                                          # beyond the tiles' line
    with torch.autocast("cuda", dtype=torch.float16):
        assert not taken()
    for make in (lambda: model.layers[1].v_proj.register_forward_hook(lambda *a: None),
                 lambda: model.layers[0].rotary_emb.register_forward_pre_hook(lambda *a: None)):
        handle = make()
        assert not taken()
        handle.remove()
    caches[1].add_seq = lambda *a: 0
    assert not taken() and taken(prefill=False, tokens=[3])
    del caches[1].add_seq
    with monkeypatch.context() as mp:
        mp.setattr(capi.Attention, "add_seq", lambda *a: 0)
        assert not taken()
    with monkeypatch.context() as mp:
        mp.setattr(model.embed_tokens, "max_norm", 1.0)
        assert not taken()
    with monkeypatch.context() as mp:
        mp.setattr(model.norm, "weight", torch.nn.Parameter(torch.ones(256, device=dev), requires_grad=False))
        assert not taken()                                                        # another type
    with monkeypatch.context() as mp:
        mp.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
        assert not taken()
    assert taken()
    with torch.enable_grad():                                                     # a gradient is wanted: not asked at all
        assert not model._adds_in_norms()
    with torch.inference_mode():
        assert model.logits([Sequence(ids)], caches, True).shape == (1, 60)


def test_refused_decode_passes_leave_every_cache_as_it_was():
    """A later layer's cache that does not fit the pass is noticed before an earlier one takes the tokens."""
    from chunk_attn.models.sequence import Sequence
    from chunk_attn.models.tiny_lm import AttentionOnlyLM
    model = AttentionOnlyLM(60, 256, 2, 3, chunk_size=32, memory_mb=8, seed=7)

    def start():
        caches, running = model.create_kv_caches(), []
        for p in (10, 31, 40):
            seq = Sequence([(t * 7 + p) % 60 for t in range(p)])
            model.logits([seq], caches, True)
            running.insert(seq.index, seq)
        for seq in running:
            seq.append(5)
        return caches, running

    def refused(caches, running, match):
        before = [c.tree.get_chunks() for c in caches]
        for _ in range(2):
            with pytest.raises(RuntimeError, match=match):
                model.logits(running, caches, False)
            assert all((a == c.tree.get_chunks()).all() for a, c in zip(before, caches))

    with torch.inference_mode():
        caches, running = start()
        caches[2].remove_seq(1)                        # other sequences in the tree
        refused(caches, running, "num of seqs")
        caches, running = start()
        want = model.logits(running, caches, False)
        caches, running = start()
        rows = caches[1].tree.get_chunks()
        first = rows[rows[:, 2] == 0]
        caches[1].ctx.refresh(first, 1, torch.cuda.current_stream().cuda_stream)     # other sequences in the tables
        refused(caches, running, "refresh first")
        caches[1].refresh_kernel_context(force=True)
        assert torch.equal(model.logits(running, caches, False), want)


@pytest.mark.parametrize("hooked", [False, True])
@pytest.mark.parametrize("over", [5, 0])               # no chunk for the prompt's end; none for its next token
def test_a_prompt_that_a_later_cache_cannot_take(hooked, over):
    """The pass fails; where the prompt stands in the caches that took it is known, to remove it there."""
    from chunk_attn import capi
    from chunk_attn.models.sequence import Sequence
    from chunk_attn.models.tiny_lm import AttentionOnlyLM
    model = AttentionOnlyLM(60, 256, 2, 2, chunk_size=32, memory_mb=8, seed=7)
    if hooked:                                         # the modules' own calls
        model.norm.register_forward_hook(lambda m, a, out: None)
    caches = model.create_kv_caches()
    caches[1] = capi.Attention(2, 128, 32, memory_mb=1, dtype=torch.float16, device=torch.device("cuda:0"))
    with torch.inference_mode():
        model.logits([Sequence([59, 58])], [caches[0], model.create_kv_caches()[1]], True)     # index 0 is taken there
        for layer in model.layers:
            layer.last_indices = None
        seq = Sequence([t % 50 for t in range(32 * caches[1].max_chunks + over)])
        with pytest.raises(RuntimeError, match="capacity reached"):
            model.logits([seq], caches, True)
    assert caches[0].tree.n_seqs == 2 and model.layers[0].last_indices == [seq.index]
    assert model.layers[1].last_indices is None
    caches[0].remove_seq(model.layers[0].last_indices[0])
    assert caches[0].tree.dump()[1][2][:2] == [59, 58]


@pytest.mark.parametrize("hidden,prompts", [
    (1024, [3] * 9), (1024, [2] * 16), (384, [5, 1, 9]),   # both numbers of rows that are normalised on their way
    (1024, [2] * 17), (1152, [7, 40])])                     # more rows, longer ones: a launch of its own
def test_norms_on_the_way_keep_every_bit(hidden, prompts):
    """Rows normalised by the projection that reads them, and sums that the output projection writes, against the
    modules' own launches, with weights and an epsilon that show in the result."""
    from chunk_attn.models.sequence import Sequence
    from chunk_attn.models.tiny_lm import AttentionOnlyLM
    runs = []
    for hooked in (False, True):
        model = AttentionOnlyLM(333, hidden, hidden // 128, 2, chunk_size=32, memory_mb=32, seed=8)
        g = torch.Generator().manual_seed(hidden)
        with torch.no_grad():
            for norm in (*model.input_norms, model.norm):
                norm.weight.copy_(torch.randn(hidden, generator=g))
                norm.eps = 0.3
        if hooked:
            model.norm.register_forward_hook(lambda m, a, out: None)
        caches, running, out = model.create_kv_caches(), [], []
        with torch.inference_mode():
            for i, n in enumerate(prompts):
                seq = Sequence([(7 * t + 50 * i) % 333 for t in range(n)])
                out.append(model.logits([seq], caches, True))
                running.insert(seq.index, seq)
            for t in range(2):
                for s, seq in enumerate(running):
                    seq.append((11 * t + 3 * s) % 333)
                out.append(model.logits(running, caches, False))
        runs.append(out)
    assert all(torch.equal(a, b) for a, b in zip(*runs)) and all(torch.isfinite(a).all() for a in runs[0])


@pytest.mark.parametrize("hidden,prompts", [(256, [40, 3]), (1024, [2] * 8), (1024, [3] * 9), (384, [1] * 16), (1024, [2] * 17), (1152, [7, 40])])
def test_the_last_norms_rows_are_in_the_scratch_with_a_head_too(hidden, prompts):
    """Where ca_model_last_rows says, after prompts and decode passes, whoever normalised them; guard rows behind stay."""
    import ctypes
    from chunk_attn import capi
    from chunk_attn.models.sequence import Sequence
    from chunk_attn.models.tiny_lm import AttentionOnlyLM
    dev, lib = torch.device("cuda:0"), capi.load()
    model = AttentionOnlyLM(60, hidden, hidden // 128, 2, chunk_size=32, memory_mb=32, seed=9)
    g = torch.Generator().manual_seed(hidden)
    with torch.no_grad():
        for norm in (*model.input_norms, model.norm):
            norm.weight.copy_(torch.randn(hidden, generator=g))

    def rows_of(caches, seqs, ids, positions, prefill, head):
        layers, kept = model._plain_pass(seqs, ids, caches, prefill, dev)
        table = (capi.ModelLayer * len(layers))(*[(cache.ctx._h, cache.tree._h, *rest) for cache, *rest in layers])
        tokens, places = sum(ids, []), sum(positions, [])
        n, i32 = len(tokens), ctypes.c_int32 * len(tokens)
        scratch = torch.full((lib.ca_model_scratch_bytes(n, hidden) // 2 + 64,), 5.0, dtype=torch.float16, device=dev)
        logits = torch.empty((len(seqs), 60), dtype=torch.float16, device=dev)
        capi._launch(dev, lib.ca_model_pass, table, len(layers), i32(*tokens), i32(*places), len(seqs), n // len(seqs), int(prefill),
                     model.embed_tokens.weight.data_ptr(), 60, model.input_norms[0].weight.data_ptr(), model.input_norms[0].eps,
                     hidden, scratch.data_ptr(), model.lm_head.weight.data_ptr() if head else None, 60 if head else 0,
                     logits.data_ptr() if head else None, (ctypes.c_int32 * len(layers))())
        assert (scratch[-64:] == 5.0).all()
        at = lib.ca_model_last_rows(n, hidden, len(seqs)) // 2
        rows = scratch[at:at + len(seqs) * hidden].view(len(seqs), hidden)
        if head:                                         # (what a pass with a head is for)
            assert torch.equal(logits, capi.linear(rows.clone(), model.lm_head.weight))
        return rows

    with torch.inference_mode():
        found = []
        for head in (False, True):
            caches, rows = model.create_kv_caches(), []
            for s, n in enumerate(prompts):
                ids = [(7 * t + 5 * s) % 60 for t in range(n)]
                rows.append(rows_of(caches, [Sequence(ids)], [ids], [list(range(n))], True, head))
            for t in range(2):
                ids = [[(11 * t + 3 * s) % 60] for s in range(len(prompts))]
                rows.append(rows_of(caches, [None] * len(prompts), ids, [[9 + t]] * len(prompts), False, head))
            found.append(rows)
        assert all(torch.equal(a, b) and torch.isfinite(a).all() for a, b in zip(*found))
