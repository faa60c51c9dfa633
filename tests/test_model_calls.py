"""The small model's and the layer's Python on the CPU: the native operators are emulated through raw addresses,
as the kernels write (past autograd, modes and hooks), and a cache that only counts stands in for the real one."""
import ctypes

import numpy as np
import pytest
import torch

from chunk_attn import capi
from chunk_attn.models.sequence import Sequence
from chunk_attn.models import tiny_lm
from chunk_attn.models.tiny_lm import AttentionOnlyLM


def raw(t):
    """The tensor's memory, with nothing of torch in between."""
    return np.ctypeslib.as_array((ctypes.c_uint16 * t.numel()).from_address(t.data_ptr())).view(np.float16).reshape(t.shape)


def normed(x, weight, eps):
    x = x.astype(np.float32)
    return (x / np.sqrt((x * x).mean(-1, keepdims=True) + eps)).astype(np.float16) * weight


class CountingCache:
    def __init__(self):
        self.n = 0

    def add_seq(self, tokens, k, v):
        self.n += 1
        return self.n - 1

    def reserve(self):
        return 0

    def refresh_kernel_context(self, force=False):
        pass


@pytest.fixture
def fused(monkeypatch):
    """Emulated operators; the list has one entry a fused add and norm."""
    calls = []

    def rms_norm(out, x, weight, eps):
        raw(out)[...] = normed(raw(x), raw(weight), eps)

    def add_rms_norm(x, residual, weight, eps):
        calls.append(x.shape)
        raw(residual)[...] = raw(residual) + raw(x)
        raw(x)[...] = normed(raw(residual), raw(weight), eps)

    monkeypatch.setattr(capi, "rms_norm", rms_norm)
    monkeypatch.setattr(capi, "add_rms_norm", add_rms_norm)
    monkeypatch.setattr(capi, "rotary_embedding", lambda *a: None)
    return calls


def model(layers=2):
    return AttentionOnlyLM(50, 32, 2, layers, max_position_embeddings=64, seed=3, device="cpu")


def logits(m):
    return m.logits([Sequence([3, 1, 4, 1, 5])], [CountingCache() for _ in m.layers], True)


def test_default_device_places_nothing_of_a_pass(fused):
    m = model()
    with torch.no_grad():
        want = logits(m)
        with torch.device("meta"):
            got = logits(m)
    assert torch.equal(got, want)


def test_no_pinned_upload_is_captured(monkeypatch):
    """A captured copy would read its staging buffer again on every replay, long after it was given back."""
    for capturing in (False, True):
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
        assert tiny_lm._pins(torch.device("cuda:0")) is not capturing
        assert not tiny_lm._pins(torch.device("cpu"))


def test_what_stands_between_a_call_and_its_kernel():
    """A default device does not; a mode that sees the operations does, alone and beside a default device."""
    class Watching(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    assert capi.plain_call()
    with torch.device("cpu"):
        assert capi.plain_call()
        with Watching():
            seen = capi.plain_call()
        assert not seen
    with Watching(), torch.device("cpu"):
        seen = capi.plain_call()
    assert not seen
    with torch.autograd.forward_ad.dual_level():
        assert not capi.plain_call()


def test_tensors_that_a_mode_saw_are_not_overwritten(fused):
    class Keeping(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            out = func(*args, **(kwargs or {}))
            if func is torch.nn.functional.linear:
                kept.append((out, out.clone()))
            return out

    m, kept = model(), []
    with torch.no_grad():
        want = logits(m)
        assert len(fused) == 2
        with Keeping():
            got = logits(m)
    assert len(kept) == 2 * 4 + 1 and all(torch.equal(a, b) for a, b in kept)
    assert torch.allclose(got, want, rtol=2e-3, atol=2e-3)              # fp16 roundings of the residual


def test_no_tangent_of_an_overwritten_tensor_reaches_the_logits(fused):
    """The norms drop tangents (they are native calls): logits of a dual output projection have none."""
    from torch.autograd import forward_ad
    m = model()
    with torch.no_grad(), forward_ad.dual_level():
        w = m.layers[1].o_proj.weight
        dual = forward_ad.make_dual(w.detach(), torch.ones_like(w))
        del m.layers[1].o_proj.weight
        m.layers[1].o_proj.weight = dual
        assert forward_ad.unpack_dual(logits(m)).tangent is None
    assert not fused


def test_replaced_classes_and_functions_are_seen(monkeypatch, fused):
    from chunk_attn import llama_layer, stock
    from chunk_attn.llama_layer import LlamaChunkAttention, RotaryEmbedding
    nn, F = torch.nn, torch.nn.functional
    checks = {nn.Linear: stock.linear_is_stock, nn.Embedding: stock.embedding_is_stock, LlamaChunkAttention: llama_layer.layer_is_stock,
              RotaryEmbedding: lambda: stock.is_stock(RotaryEmbedding, llama_layer._ROTARY_FORWARD),
              tiny_lm.RMSNorm: lambda: stock.is_stock(tiny_lm.RMSNorm, tiny_lm._NORM_FORWARD)}
    m = model()

    def seen():
        """The classes found changed; whether the model still overwrites."""
        with torch.no_grad():
            return [cls for cls, check in checks.items() if not check()], m._adds_in_norms()

    assert seen() == ([], True)
    for cls in checks:
        with monkeypatch.context() as mp:
            forward = cls.forward
            mp.setattr(cls, "forward", lambda *a: forward(*a))
            assert seen() == ([cls], cls is RotaryEmbedding)
    for name in ("__call__", "_call_impl"):
        with monkeypatch.context() as mp:
            mp.setattr(nn.Module, name, lambda *a, **k: None)
            assert seen() == (list(checks), False)
    for name, cls in (("linear", nn.Linear), ("embedding", nn.Embedding)):
        with monkeypatch.context() as mp:
            mp.setattr(F, name, lambda *a: None)
            assert seen() == ([cls], False)
    assert stock._at_home(seen, nn) is None and stock._at_home(F.embedding, F) is F.embedding
    cache = object.__new__(capi.Attention)
    assert capi.is_plain_cache(cache) and not capi.is_plain_cache(CountingCache())
    with monkeypatch.context() as mp:
        mp.setattr(capi.Attention, "forward", lambda self, q: q)
        assert not capi.is_plain_cache(cache)
    cache.append_token_rotary = lambda *a: None
    assert not capi.is_plain_cache(cache)


def test_tables_that_only_the_operator_takes():
    """A rotary table put in by the user: narrower rows or an odd address are the operator's, not the kernels'."""
    from chunk_attn.llama_layer import LlamaChunkAttention
    layer = LlamaChunkAttention(256, 2, max_position_embeddings=8, device="cpu")
    flat = torch.zeros(8 * 128 + 1, dtype=torch.float16)
    assert layer._plain_rotary(flat.device) is layer.rotary_emb.cos_sin_cache
    for table, plain in ((flat[:-1].view(8, 128), True), (flat[1:].view(8, 128), False), (flat[:512].view(8, 64), False)):
        layer.rotary_emb.cos_sin_cache = table
        assert (layer._plain_rotary(flat.device) is table) == plain


# us on one GPU (MI355X), weights from memory
@pytest.mark.parametrize("rows,n_in,n_out,here,library,pays", [
    (2048, 128, 128, 3.1, 4.2, True), (1024, 512, 512, 5.8, 6.1, True), (252, 1024, 1024, 4.4, 8.0, True),
    (1024, 1024, 1024, 8.8, 9.0, True), (1536, 1024, 1024, 15.6, 9.9, False), (512, 1536, 1536, 10.9, 9.3, True),
    (1024, 1536, 1536, 20.2, 13.0, False), (512, 2048, 2048, 13.7, 11.4, True), (16, 4096, 4096, 8.3, 9.0, True),
    (252, 4096, 4096, 19.7, 19.2, True), (320, 4096, 4096, 34.0, 22.4, False), (128, 5120, 5120, 30.2, 25.0, True),
    (252, 5120, 5120, 41.9, 27.4, False), (16, 8192, 8192, 26.2, 22.0, True), (48, 8192, 8192, 46.4, 25.6, False),
    (65, 1024, 4000, 7.4, 8.5, True), (512, 1024, 4000, 20.0, 11.7, False), (128, 1024, 8000, 10.6, 9.6, True),
    (160, 1024, 8000, 17.4, 10.4, False), (252, 1024, 8000, 19.8, 11.2, False), (32, 1024, 32000, 21.2, 23.6, True),
    (252, 1024, 32000, 69.3, 25.4, False), (16, 4096, 32000, 58.6, 57.7, True), (252, 4096, 32000, 193.8, 75.4, False),
    (16, 4096, 11008, 23.7, 20.8, True), (64, 4096, 11008, 37.9, 27.5, False)])
def test_projections_are_computed_here_while_the_host_gains_more(rows, n_in, n_out, here, library, pays):
    """A library call costs the host 9 us more than one here."""
    assert capi.projection_pays(rows, n_in, n_out) == pays
    assert here <= library + 9 if pays else here > library + 5


class AnyGpu:
    """A GPU that every tensor lies on."""
    type = "cuda"
    __hash__ = None

    def __eq__(self, other):
        return True

    def __ne__(self, other):
        return False


def hide_projection(m, mp):
    m.layers[1].__dict__["q_proj"] = lambda x: x


def hide_output_projection(m, mp):
    m.layers[0].__dict__["o_proj"] = m.layers[1].o_proj


def function_for_a_deleted_projection(m, mp):
    del m.layers[0].v_proj
    m.layers[0].v_proj = torch.relu                            # a builtin: no dictionary of its own


def hide_projections_of_the_class(m, mp):
    mp.setattr(tiny_lm.LlamaChunkAttention, "k_proj", staticmethod(lambda x: x), raising=False)


def hide_weight(m, mp):
    m.layers[0].k_proj.__dict__["weight"] = m.layers[1].k_proj.weight


def hide_bias(m, mp):
    m.layers[0].o_proj.__dict__["bias"] = torch.ones(128, dtype=torch.float16)


def hide_norm_weight(m, mp):
    m.input_norms[1].__dict__["weight"] = m.norm.weight


def hide_rotary_table(m, mp):
    m.layers[1].rotary_emb.__dict__["cos_sin_cache"] = torch.zeros(64, 128, dtype=torch.float16)


@pytest.mark.parametrize("hide", [
    hide_projection, hide_output_projection, function_for_a_deleted_projection, hide_projections_of_the_class, hide_weight,
    hide_bias, hide_norm_weight, hide_rotary_table])
def test_native_pass_sees_what_hides_a_registered_module(monkeypatch, hide):
    """Python finds an attribute of the object, and of its class, before the module or parameter of that name."""
    import types
    gpu = AnyGpu()
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(capi, "is_plain_cache", lambda c: True)
    monkeypatch.setattr(capi, "is_plain_cache_to_fill", lambda c: True)
    caches = [types.SimpleNamespace(d_head=128, n_heads=1, device=gpu)] * 2

    def taken(m):
        return [m._plain_pass([None], [[1, 2][:n]], caches, n == 2, gpu) is not None for n in (1, 2)]

    with torch.no_grad():
        m = AttentionOnlyLM(50, 128, 1, 2, max_position_embeddings=64, seed=3, device="cpu")
        assert taken(m) == [True, True]
        hide(m, monkeypatch)
        assert taken(m) == [False, False]
