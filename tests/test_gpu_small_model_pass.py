"""The small model's native pass against its modules' own calls."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,layers,prompts,chunk,vocab", [
    (128, 1, [1, 5], 32, 40), (1024, 3, [449, 30, 449], 64, 300), (512, 2, [900, 65, 64, 63], 128, 1001)])
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
