"""The caller of the decode path: one Llama attention layer over the prefix-tree KV cache.

Mirrors the reference's `LlamaChunkAttention`
(src/chunk_attn/models/llama_hf/modeling_llama.py:16-113) and its rotary module
(src/chunk_attn/models/llama_hf/rotary_embedding_vllm.py:43-147) with the same argument
meaning.  Up to some thousand rows the three input projections and the rotary embedding are one
launch, in the decode branch the KV append too; for more the projections are plain torch matmuls, and
the rotary embedding of a decode step's query/key rows and the KV append are one launch
(`Attention.append_token_rotary`).
Weights are whatever the caller loads; tests use seeded random ones.
"""
from __future__ import annotations

import math
from typing import List, Optional, Sequence

import torch
from torch import nn

from . import capi, stock


class RotaryEmbedding(nn.Module):
    """cos/sin cache [max_position, rotary_dim] (fp32 math, stored fp16) and the in-place operator."""

    def __init__(self, head_size: int, rotary_dim: int, max_position_embeddings: int = 10240,
                 base: float = 10000.0, is_neox_style: bool = True, device="cuda"):
        super().__init__()
        self.head_size, self.rotary_dim = head_size, rotary_dim
        self.max_position_embeddings, self.base, self.is_neox_style = max_position_embeddings, base, is_neox_style
        inv_freq = 1.0 / (base ** (torch.arange(0, rotary_dim, 2, dtype=torch.float, device=device) / rotary_dim))
        t = torch.arange(max_position_embeddings, dtype=torch.float, device=device)
        freqs = torch.einsum("i,j -> ij", t, inv_freq)
        cache = torch.cat((freqs.cos(), freqs.sin()), dim=-1).to(torch.float16)
        self.register_buffer("cos_sin_cache", cache.contiguous(), persistent=False)

    def forward(self, positions: torch.Tensor, query: torch.Tensor, key: torch.Tensor):
        capi.rotary_embedding(positions, query, key, self.head_size, self.cos_sin_cache, self.is_neox_style)
        return query, key


_ROTARY_FORWARD = RotaryEmbedding.forward


def plain_rotaries(layers, device: torch.device) -> Optional[List[torch.Tensor]]:
    """The layers' rotary tables, if every one is as LlamaChunkAttention._plain_rotary says."""
    return capi.modules.rotary_tables(layers, RotaryEmbedding, device) if stock.is_stock(RotaryEmbedding, _ROTARY_FORWARD) else None


class LlamaChunkAttention(nn.Module):
    """q/k/v projections -> rotary -> (prefill: causal attention + add_seq | decode: append +
    chunk attention) -> output projection."""

    def __init__(self, hidden_size: int, num_heads: int, max_position_embeddings: int = 10240,
                 rope_base: float = 10000.0, dtype=torch.float16, device="cuda"):
        super().__init__()
        if hidden_size % num_heads:
            raise ValueError(f"hidden_size must be divisible by num_heads (got `hidden_size`: {hidden_size}"
                             f" and `num_heads`: {num_heads}).")
        self.hidden_size, self.num_heads, self.head_dim = hidden_size, num_heads, hidden_size // num_heads
        kw = dict(bias=False, dtype=dtype, device=device)
        self.q_proj = nn.Linear(hidden_size, hidden_size, **kw)
        self.k_proj = nn.Linear(hidden_size, hidden_size, **kw)
        self.v_proj = nn.Linear(hidden_size, hidden_size, **kw)
        self.o_proj = nn.Linear(hidden_size, hidden_size, **kw)
        self.rotary_emb = RotaryEmbedding(self.head_dim, self.head_dim, max_position_embeddings, rope_base,
                                          True, device)

    def forward(self, hidden_states: torch.Tensor, seqs: List[Sequence[int]], position_ids: torch.Tensor,
                kv_cache: capi.Attention, prefill: bool) -> torch.Tensor:
        """hidden_states [n_seqs, n_tokens, hidden]; seqs: each sequence's token ids so far (the
        new token last); position_ids int64 [n_seqs, n_tokens].  Prefill inserts the sequences
        into kv_cache (their cache indices are returned in self.last_indices); decode expects
        batch row i to be cache sequence i."""
        batch, n_tokens, d_hidden = hidden_states.shape
        projections = (self.q_proj, self.k_proj, self.v_proj)
        own_output = own_input = False                 # which projections the framework's own kernels compute
        rows = batch * n_tokens
        few_rows = capi.projection_pays(rows, d_hidden, d_hidden)
        if self.head_dim == 128 and (few_rows or prefill and capi.shared_tiles_pay(rows, d_hidden, d_hidden, 3)) and \
                stock.linear_is_stock():
            limit = hidden_states.numel()              # the two rules have looked at the size
            table = self._plain_rotary(hidden_states.device)
            own_output = table is not None and (few_rows or capi.shared_tiles_pay(rows, d_hidden, d_hidden, 1)) and \
                capi._projection_takes(hidden_states, *projections, self.o_proj, limit=limit)
            own_input = own_output or table is not None and capi._projection_takes(hidden_states, *projections, limit=limit)
        if own_input:
            weights = [p.weight for p in projections]
        if own_input and not prefill and capi.is_plain_cache(kv_cache):     # other caches have append_token_rotary only
            assert n_tokens == 1
            step = ([s[-1] for s in seqs], hidden_states, *weights)
            rotary = (table, position_ids.reshape(batch).contiguous())
            if own_output:
                return kv_cache._layer_decode(*step, self.o_proj.weight, *rotary).view(batch, 1, -1)
            q3 = kv_cache._project_append_rotary(*step, *rotary)
            return self._output(kv_cache.forward(q3).view(batch, 1, d_hidden), kv_cache, False)
        if own_input and prefill:
            q, k, v = capi._qkv_rotary(hidden_states, *weights, position_ids.contiguous(), table)
        else:
            q = self.q_proj(hidden_states)
            k = self.k_proj(hidden_states)
            v = self.v_proj(hidden_states)
        if prefill:
            if not own_input:
                q, k = self.rotary_emb(position_ids.contiguous(), q, k)
            shape = (batch, n_tokens, self.num_heads, self.head_dim)
            q4, k4, v4 = q.view(shape), k.view(shape), v.view(shape)
            takes = hidden_states.dtype == torch.float16 and capi.causal_attention_takes(q4, k4, v4)
            both = kv_cache._prefill_attention(seqs, q4, k4, v4) if takes and capi.is_plain_cache_to_fill(kv_cache) else None
            if both is not None:
                attn_output, self.last_indices = both[0].view(batch, n_tokens, d_hidden), both[1]
            elif takes:
                attn_output = capi._causal_attention(q4, k4, v4).view(batch, n_tokens, d_hidden)
            else:
                # what the kernel does not take (a gradient is wanted, another head size): plain fp32 torch math
                qh, kh, vh = (t.transpose(1, 2).float() for t in (q4, k4, v4))
                scores = qh @ kh.transpose(-1, -2) / math.sqrt(self.head_dim)
                future = torch.ones(n_tokens, n_tokens, dtype=torch.bool, device=scores.device).triu(1)
                attn = torch.softmax(scores.masked_fill(future, float("-inf")), dim=-1) @ vh
                attn_output = attn.transpose(1, 2).reshape(batch, n_tokens, d_hidden).to(hidden_states.dtype)
            if both is None:
                self.last_indices = [kv_cache.add_seq(list(seqs[i]), k4[i].contiguous(), v4[i].contiguous())
                                     for i in range(batch)]
        else:
            assert n_tokens == 1
            shape = (batch, self.num_heads, self.head_dim)
            q3, k3, v3 = q.view(shape), k.view(shape), v.view(shape)
            kv_cache.append_token_rotary([s[-1] for s in seqs], q3, k3, v3, self.rotary_emb.cos_sin_cache,
                                         self.rotary_emb.is_neox_style, position_ids.reshape(batch).contiguous())
            attn_output = kv_cache.forward(q3).view(batch, 1, d_hidden)
            # a cache of another class may return anything: another type, a subclass, something with a gradient
            own_output = own_output and capi._projection_takes(attn_output, self.o_proj)
        return self._output(attn_output, kv_cache, own_output)

    def _plain_rotary(self, device: torch.device) -> Optional[torch.Tensor]:
        """The rotary module's table, if the module is the one this layer was built with, over whole heads, nothing
        hangs on it or hides its table, and the projection kernels read such a table (the operator takes narrower ones and any
        alignment)."""
        tables = plain_rotaries((self,), device)
        return tables[0] if tables else None

    def _output(self, attn_output: torch.Tensor, kv_cache: capi.Attention, own: bool) -> torch.Tensor:
        output = capi._linear(attn_output, self.o_proj.weight) if own else self.o_proj(attn_output)
        kv_cache.reserve()
        kv_cache.refresh_kernel_context(force=False)
        return output


_LAYER_FORWARD = LlamaChunkAttention.forward


def layer_is_stock() -> bool:
    return stock.is_stock(LlamaChunkAttention, _LAYER_FORWARD)
