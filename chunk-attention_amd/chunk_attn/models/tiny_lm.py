"""A small attention-only language model over the prefix-tree KV caches: embedding, a stack of
pre-norm `LlamaChunkAttention` layers with residuals, final norm and output head.  It has the
call signature of the reference's `LlamaForCausalLM.forward(seqs, kv_caches, prefill)`
(src/chunk_attn/models/llama_hf/modeling_llama.py:288-299, 206-235) and exists to drive the
scheduler and the decode path end to end with seeded weights; it is not a trained model.
"""
from __future__ import annotations

import array
import math
from typing import List, Optional

import torch
from torch import nn

from .. import capi, stock
from ..llama_layer import LlamaChunkAttention, layer_is_stock, plain_rotaries
from .sequence import Sequence


class RMSNorm(nn.Module):
    def __init__(self, hidden_size: int, eps: float = 1e-6, dtype=torch.float16, device="cuda"):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(hidden_size, dtype=dtype, device=device))
        self.eps = eps

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        x = x.contiguous()
        out = torch.empty_like(x)
        capi.rms_norm(out, x, self.weight, self.eps)
        return out


_NORM_FORWARD = RMSNorm.forward
_HOST = torch.device("cpu")
_PROJECTIONS = ("q_proj", "k_proj", "v_proj", "o_proj")


def _addresses(parameters, shape, device: torch.device) -> Optional[List[int]]:
    """Of parameters that kernels can read by their address; None if one is not."""
    return capi.modules.parameter_addresses(parameters, nn.Parameter, shape, device)


def _pins(device: torch.device) -> bool:
    """Whether ids for `device` go through pinned memory.  Not under stream capture: a replay would read whatever
    the staging buffer holds by then; the copy from ordinary memory is refused there."""
    return device.type == "cuda" and not torch.cuda.is_current_stream_capturing()


class AttentionOnlyLM(nn.Module):
    def __init__(self, vocab_size: int, hidden_size: int, num_heads: int, num_layers: int,
                 max_position_embeddings: int = 4096, chunk_size: int = 64, memory_mb: int = 256,
                 seed: int = 0, dtype=torch.float16, device="cuda"):
        super().__init__()
        self.vocab_size, self.hidden_size, self.num_heads = vocab_size, hidden_size, num_heads
        self.chunk_size, self.memory_mb, self.device = chunk_size, memory_mb, torch.device(device)
        self.embed_tokens = nn.Embedding(vocab_size, hidden_size, dtype=dtype, device=device)
        self.layers = nn.ModuleList([LlamaChunkAttention(hidden_size, num_heads, max_position_embeddings,
                                                         dtype=dtype, device=device) for _ in range(num_layers)])
        self.input_norms = nn.ModuleList([RMSNorm(hidden_size, dtype=dtype, device=device) for _ in range(num_layers)])
        self.norm = RMSNorm(hidden_size, dtype=dtype, device=device)
        self.lm_head = nn.Linear(hidden_size, vocab_size, bias=False, dtype=dtype, device=device)
        g = torch.Generator().manual_seed(seed)
        with torch.no_grad():
            self.embed_tokens.weight.copy_(torch.randn(vocab_size, hidden_size, generator=g))
            self.lm_head.weight.copy_(torch.randn(vocab_size, hidden_size, generator=g) / math.sqrt(hidden_size))
            for layer in self.layers:
                for p in (layer.q_proj, layer.k_proj, layer.v_proj, layer.o_proj):
                    p.weight.copy_(torch.randn(hidden_size, hidden_size, generator=g) / math.sqrt(hidden_size))

    def create_kv_caches(self) -> List[capi.Attention]:
        """One cache per layer, same configuration (reference modeling_llama.py:252-270)."""
        dev = self.device if self.device.index is not None else torch.device("cuda", torch.cuda.current_device())
        return [capi.Attention(n_heads=self.num_heads, d_head=self.hidden_size // self.num_heads,
                               chunk_size=self.chunk_size, memory_mb=self.memory_mb, share_prefix=True,
                               tpp_threshold=1, dtype=torch.float16, device=dev) for _ in self.layers]

    def logits(self, seqs: List[Sequence], kv_caches, prefill: bool) -> torch.Tensor:
        """[n_seqs, vocab] logits of every sequence's last position."""
        if prefill:
            lens = {len(s) for s in seqs}
            if len(lens) != 1:
                raise ValueError("prefill takes prompts of one length at a time")
            input_ids = [list(s.tokens) for s in seqs]
            position_ids = [list(range(len(s))) for s in seqs]
        else:
            input_ids = [[s[-1]] for s in seqs]
            position_ids = [[len(s) - 1] for s in seqs]
        embedding = self.embed_tokens.weight
        dev = embedding.device
        joined = self._adds_in_norms()
        plain = self._plain_pass(seqs, input_ids, kv_caches, prefill, dev) if joined else None
        if plain is not None:
            layers, kept = plain                       # (kept to the end of the call: addresses alone hold nothing)
            lm_head, first = self.lm_head, self.input_norms[0]
            head = lm_head.weight if capi.projection_pays(len(seqs), self.hidden_size, self.vocab_size) and \
                capi._linears_are_plain(self.hidden_size, dev, (lm_head,)) else None
            index = []
            try:
                out = capi._model_pass(layers, [t for ids in input_ids for t in ids], [p for pos in position_ids for p in pos],
                                       len(seqs), prefill, embedding, first.weight, first.eps, head, index)
            finally:                                   # a pass that failed has filled the caches in front of that layer
                for layer, idx in zip(self.layers, index) if prefill else ():
                    if idx >= 0:
                        layer.last_indices = [idx]
                        seqs[0].index = idx
            return out if head is not None else self.lm_head(out)
        # one upload, from pinned memory: the host does not wait for what the GPU still has to do (the device is
        # named: only host memory can be pinned, whatever the default device is)
        pinned = _pins(dev)
        ids, pos = torch.tensor([input_ids, position_ids], dtype=torch.int64, device=_HOST,
                                pin_memory=pinned).to(dev, non_blocking=pinned)
        hidden = self.embed_tokens(ids)
        token_lists = [s.tokens for s in seqs]
        normed = self.input_norms[0](hidden) if len(self.layers) else None
        for i, layer in enumerate(self.layers):
            out = layer(normed, token_lists, pos, kv_caches[i], prefill)
            if prefill:
                for s, idx in zip(seqs, layer.last_indices):
                    s.index = idx
            final = i + 1 == len(self.layers)
            norm = self.norm if final else self.input_norms[i + 1]
            if final:   # from here on the last positions alone
                out, hidden = out[:, -1], hidden[:, -1]
            if joined:  # hidden += out, out = norm(hidden): one launch over both, the same bits
                out, hidden = out.contiguous(), hidden.contiguous()
                capi.add_rms_norm(out, hidden, norm.weight, norm.eps)
                normed = out
            else:
                hidden = hidden + out
                normed = norm(hidden)
        last = self.norm(hidden[:, -1]) if normed is None else normed
        if capi.projection_pays(len(seqs), self.hidden_size, self.vocab_size) and stock.linear_is_stock() and \
                capi._projection_takes(last, self.lm_head):
            return capi._linear(last, self.lm_head.weight)
        return self.lm_head(last)

    def _plain_pass(self, seqs, input_ids, kv_caches, prefill: bool, dev: torch.device) -> Optional[tuple]:
        """(the layers as capi._model_pass takes them, what their addresses are of), if the pass is one that the native call
        computes as the modules would (given _adds_in_norms): a decode step or one prompt, every layer's projections its
        own kernels' business, caches and parameters plain, and no capture, under which ids are not uploaded either."""
        hidden, n = self.hidden_size, len(self.layers)
        if n == 0 or len(kv_caches) < n or not seqs or not input_ids[0] or (prefill and len(seqs) != 1) or dev.type != "cuda" or \
                torch.cuda.is_current_stream_capturing():
            return None
        rows = len(seqs) * len(input_ids[0])
        if not (capi.projection_pays(rows, hidden, hidden) or
                prefill and capi.shared_tiles_pay(rows, hidden, hidden, 3) and capi.shared_tiles_pay(rows, hidden, hidden, 1)):
            return None
        try:
            array.array("i", [t for ids in input_ids for t in ids])
        except (TypeError, OverflowError):             # ids that are no 32-bit numbers: torch's business
            return None
        norms, modules = (*self.input_norms, self.norm), list(self.layers)
        gains = [None if "weight" in m.__dict__ else m._parameters.get("weight") for m in norms]
        norm_weights, embedding = _addresses(gains, (hidden,), dev), self.embed_tokens
        if len(norms) != n + 1 or embedding.max_norm is not None or norm_weights is None or \
                _addresses((embedding.weight,), (self.vocab_size, hidden), dev) is None:
            return None
        # (by the modules' own dictionaries: __getattr__ costs as much as a launch here, a few dozen times a pass; what
        # hides a registered module, on the object or its class, is what the layer calls)
        if not vars(LlamaChunkAttention).keys().isdisjoint(_PROJECTIONS) or \
                not all([layer.__dict__.keys().isdisjoint(_PROJECTIONS) for layer in modules]):
            return None
        weights = capi.plain_weights(hidden, hidden, dev, [own.get(name) for own in [layer._modules for layer in modules] for name in _PROJECTIONS])
        if weights is None:
            return None
        tables = plain_rotaries(modules, dev)
        if tables is None:
            return None
        plain_cache = capi.is_plain_cache_to_fill if prefill else capi.is_plain_cache
        addresses, tensors = weights
        layers, kept = [], (tensors, gains, tables)
        for i, (layer, cache, table) in enumerate(zip(modules, kv_caches, tables)):
            heads = layer.num_heads
            if layer.head_dim != 128 or heads * 128 != hidden or not plain_cache(cache) or cache.d_head != 128 or \
                    cache.n_heads != heads or cache.device != dev:
                return None
            layers.append((cache, *addresses[4 * i:4 * i + 4], table.data_ptr(), norm_weights[i + 1], table.shape[0], norms[i + 1].eps))
        return layers, kept

    def _adds_in_norms(self) -> bool:
        """A layer's residual is added in the norm behind it, in place: nothing may want the tensors it overwrites
        (a gradient, a hook, a mode that sees them, a forward-mode tangent of them), and the norms must be the plain
        ones."""
        bare, layers = capi.modules.all_bare, list(self.layers)
        return capi.plain_call() and not torch.is_grad_enabled() and \
            stock.embedding_is_stock() and stock.linear_is_stock() and layer_is_stock() and \
            stock.is_stock(RMSNorm, _NORM_FORWARD) and \
            not torch.nn.modules.module._has_any_global_hook() and capi.is_bare(self.embed_tokens, nn.Embedding) and \
            bare(LlamaChunkAttention, layers) and capi.modules.children_bare(nn.Linear, layers, "o_proj") and \
            bare(RMSNorm, (*self.input_norms, self.norm))

    @torch.no_grad()
    def forward(self, seqs: List[Sequence], kv_caches, prefill: bool) -> List[int]:
        return torch.argmax(self.logits(seqs, kv_caches, prefill), dim=-1).tolist()
