"""A small attention-only language model over the prefix-tree KV caches: embedding, a stack of
pre-norm `LlamaChunkAttention` layers with residuals, final norm and output head.  It has the
call signature of the reference's `LlamaForCausalLM.forward(seqs, kv_caches, prefill)`
(src/chunk_attn/models/llama_hf/modeling_llama.py:288-299, 206-235) and exists to drive the
scheduler and the decode path end to end with seeded weights; it is not a trained model.
"""
from __future__ import annotations

import math
from typing import List

import torch
from torch import nn

from .. import capi, stock
from ..llama_layer import LlamaChunkAttention, layer_is_stock
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
        dev = self.embed_tokens.weight.device
        # one upload, from pinned memory: the host does not wait for what the GPU still has to do (the device is
        # named: only host memory can be pinned, whatever the default device is)
        pinned = _pins(dev)
        ids, pos = torch.tensor([input_ids, position_ids], dtype=torch.int64, device=_HOST,
                                pin_memory=pinned).to(dev, non_blocking=pinned)
        hidden = self.embed_tokens(ids)
        token_lists = [s.tokens for s in seqs]
        joined = self._adds_in_norms()
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

    def _adds_in_norms(self) -> bool:
        """A layer's residual is added in the norm behind it, in place: nothing may want the tensors it overwrites
        (a gradient, a hook, a mode that sees them, a forward-mode tangent of them), and the norms must be the plain
        ones."""
        return capi.plain_call() and not torch.is_grad_enabled() and \
            stock.embedding_is_stock() and stock.linear_is_stock() and layer_is_stock() and \
            stock.is_stock(RMSNorm, _NORM_FORWARD) and \
            not torch.nn.modules.module._has_any_global_hook() and capi.is_bare(self.embed_tokens, nn.Embedding) and \
            all([capi.is_bare(m, LlamaChunkAttention) and capi.is_bare(m.o_proj, nn.Linear) for m in self.layers]) and \
            all([capi.is_bare(m, RMSNorm) for m in (*self.input_norms, self.norm)])

    @torch.no_grad()
    def forward(self, seqs: List[Sequence], kv_caches, prefill: bool) -> List[int]:
        return torch.argmax(self.logits(seqs, kv_caches, prefill), dim=-1).tolist()
