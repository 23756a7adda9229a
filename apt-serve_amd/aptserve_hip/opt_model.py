"""Minimal OPT decoder stack over the hybrid cache — the GPU side of a serving step.

Mirrors ``OPTDecoderLayer.forward`` / ``OPTDecoder.forward``
(additional_designs/model_executor/models/aptserve_opt.py:179-212, 266-290) for the
pre-LayerNorm OPT variants (``do_layer_norm_before=True``: 125m, 1.3b ... 175b): the hidden
state cached for a hidden-cached sequence is the output of ``self_attn_layer_norm``, i.e.
the input of ``qkv_proj``.  Weights are random-initialised from a locally built config
(no checkpoint, no tokenizer).  Attention, the q/kv projections, the cache traffic, fc1 and
fc2 run on this library's kernels, and so does every (residual add, LayerNorm) pair
(``ops.add_layer_norm``: one launch instead of two element-wise ones; ``fused_norm=False``
keeps the plain PyTorch-ROCm ops); ReLU and the embedding lookup are PyTorch-ROCm ops.
"""

from __future__ import annotations

from dataclasses import dataclass
from typing import Dict, List, Optional

import torch
import torch.nn.functional as F

from . import ops
from .backend import HybridOPTAttention, phase
from .metadata import HybridAttentionMetadata


@dataclass
class OPTConfig:
    hidden_size: int = 5120
    num_attention_heads: int = 40
    num_hidden_layers: int = 40
    ffn_dim: int = 20480
    vocab_size: int = 50272
    max_position_embeddings: int = 2048

    @staticmethod
    def opt_13b() -> "OPTConfig":
        return OPTConfig()

    @staticmethod
    def opt_125m() -> "OPTConfig":
        return OPTConfig(768, 12, 12, 3072, 50272, 2048)


#: Bytes added to the row pitch of a matrix whose rows are a multiple of 2 KiB long, but not a power of two.  At such a
#: pitch the 128-byte pieces that a k-tile takes of many rows meet in few channels of the memory side: fc2 of 361 rows
#: (rows of 40 KiB) takes 131 us, 107 with its weight at the longer pitch and 92 with the activations as well, fc1 86 and
#: 82, qkv 83 and 78 (rows of 10 KiB), a whole prompt step of 361 tokens 14.15 ms and 12.62.  Rows of 4, 8 or 16 KiB are read
#: no faster at a longer pitch.  Products of at most 48 rows stream whole rows and care little: fc2 of 5 rows 37.5 us and
#: 38.2, a decode step of 5 sequences 7.28 ms and 7.29, of 16 (20 layers) 4.72 and 4.64.
_PITCH_PAD = 128


def _row_pitch(k: int, dtype) -> int:
    row = k * dtype.itemsize
    return k + (_PITCH_PAD // dtype.itemsize if row % 2048 == 0 and row & (row - 1) else 0)


def row_pitched(n: int, k: int, dtype, device) -> torch.Tensor:
    """An uninitialised ``[n, k]`` matrix at the row pitch the products of this library read fastest; every operator
    takes it in place of a contiguous matrix.  (One call, as ``torch.empty`` is: prompt steps of small models are bound by
    the host.)"""
    return torch.empty_strided((n, k), (_row_pitch(k, dtype), 1), dtype=dtype, device=device)


def lay_out_weights(weights: Dict[str, torch.Tensor]) -> Dict[str, torch.Tensor]:
    """Puts the layers' matrices at the pitch of :func:`row_pitched`: to be called once, on loaded (contiguous) weights
    and before a model is built from them.  Works in the given dict, one matrix at a time, and returns it; what holds on
    to a replaced tensor keeps the old memory.  A loader that fills :func:`row_pitched` matrices has no need of it."""
    for name, w in weights.items():
        if name.startswith("layers.") and w.dim() == 2 and w.stride() == (w.size(1), 1) and w.size(1) != _row_pitch(
                w.size(1), w.dtype):
            weights[name] = row_pitched(*w.shape, w.dtype, w.device).copy_(w.detach())
    return weights


def random_weights(cfg: OPTConfig, seed: int, device, dtype=torch.float16, layers: Optional[int] = None
                   ) -> Dict[str, torch.Tensor]:
    """N(0, 0.02) matrices, N(0, 0.02) biases, LayerNorm gains near 1 — generated on ``device``; the layers'
    matrices lie at the pitch of :func:`row_pitched`, as a loader would put them (or :func:`lay_out_weights`)."""
    g = torch.Generator(device=device).manual_seed(seed)
    Hd, F_, L = cfg.hidden_size, cfg.ffn_dim, cfg.num_hidden_layers if layers is None else layers

    def values(*shape, std=0.02, mean=0.0):
        return torch.randn(*shape, generator=g, device=device, dtype=torch.float32) * std + mean

    def n(*shape, **kw):
        return values(*shape, **kw).to(dtype)

    def m(*shape):
        return row_pitched(*shape, dtype, device).copy_(values(*shape))
    w = {"embed_tokens": n(cfg.vocab_size, Hd), "embed_positions": n(cfg.max_position_embeddings + 2, Hd),
         "final_ln_w": n(Hd, std=0.02, mean=1.0), "final_ln_b": n(Hd)}
    for i in range(L):
        p = f"layers.{i}."
        w.update({p + "attn_ln_w": n(Hd, mean=1.0), p + "attn_ln_b": n(Hd),
                  p + "qkv_w": m(3 * Hd, Hd), p + "qkv_b": n(3 * Hd),
                  p + "out_w": m(Hd, Hd), p + "out_b": n(Hd),
                  p + "final_ln_w": n(Hd, mean=1.0), p + "final_ln_b": n(Hd),
                  p + "fc1_w": m(F_, Hd), p + "fc1_b": n(F_), p + "fc2_w": m(Hd, F_), p + "fc2_b": n(Hd)})
    return w


class HybridOPTDecoderLayer:
    def __init__(self, cfg: OPTConfig, w: Dict[str, torch.Tensor], prefix: str, **attn_kw) -> None:
        self.w, self.p, self.cfg = w, prefix, cfg
        self.self_attn = HybridOPTAttention(cfg.hidden_size, cfg.num_attention_heads, w[prefix + "qkv_w"],
                                            w[prefix + "qkv_b"], w[prefix + "out_w"], w[prefix + "out_b"], **attn_kw)

    def _fc1(self, x):
        """fc1 with its ReLU (stored by fc1's own epilogue)."""
        w, p = self.w, self.p
        # more rows than the weight-streaming products take: the tile kernel reads x by k-tiles too
        out = row_pitched(x.size(0), w[p + "fc1_w"].size(0), x.dtype, x.device) if x.size(0) > 48 else None
        return ops.linear_nt(x, w[p + "fc1_w"], w[p + "fc1_b"], out=out, relu=True)

    def _mlp(self, x):
        with phase("projections"):
            return ops.linear_nt(self._fc1(x), self.w[self.p + "fc2_w"], self.w[self.p + "fc2_b"])

    def forward(self, hidden_states, kv_cache, shared_cache, md: HybridAttentionMetadata):
        """additional_designs/model_executor/models/aptserve_opt.py:179-212 with plain element-wise ops."""
        w, p, Hd = self.w, self.p, self.cfg.hidden_size
        residual = hidden_states
        hidden_states = F.layer_norm(hidden_states, (Hd,), w[p + "attn_ln_w"], w[p + "attn_ln_b"])
        hidden_states = self.self_attn(hidden_states, kv_cache, shared_cache, md)
        hidden_states = residual + hidden_states
        residual = hidden_states
        hidden_states = F.layer_norm(hidden_states, (Hd,), w[p + "final_ln_w"], w[p + "final_ln_b"])
        return residual + self._mlp(hidden_states)

    def forward_fused_norm(self, residual, normed, kv_cache, shared_cache, md, next_ln_w, next_ln_b):
        """The same layer with every (residual add, LayerNorm) pair in one launch, which also adds the K parts of the
        product in front of it where there are any.  ``normed`` is this layer's
        ``self_attn_layer_norm`` of ``residual`` (computed by the previous layer's last launch); returns the
        layer's output and the NEXT norm of it (the next layer's ``self_attn_layer_norm``, or the decoder's
        final one)."""
        w, p = self.w, self.p
        a = self.self_attn
        if type(a).__call__ is not HybridOPTAttention.forward or getattr(self._mlp, "__func__", None) is not _OWN_MLP:
            # something else in place of the attention or of the MLP is called as a whole: its last product is its own
            normed, residual = ops.add_layer_norm(a(normed, kv_cache, shared_cache, md), residual, w[p + "final_ln_w"],
                                                  w[p + "final_ln_b"])
            normed, residual = ops.add_layer_norm(self._mlp(normed), residual, next_ln_w, next_ln_b)
            return residual, normed
        attn = a.attend(normed, kv_cache, shared_cache, md)
        with phase("projections"):
            normed, residual = ops.linear_add_layer_norm(attn, a.out_weight, a.out_bias, residual, w[p + "final_ln_w"],
                                                         w[p + "final_ln_b"])
            normed, residual = ops.linear_add_layer_norm(self._fc1(normed), w[p + "fc2_w"], w[p + "fc2_b"], residual,
                                                         next_ln_w, next_ln_b)
        return residual, normed

    __call__ = forward


_OWN_MLP = HybridOPTDecoderLayer._mlp


class HybridOPTModel:
    """``weights`` are used as they lie: matrices at the pitch of :func:`row_pitched` make prompt steps faster."""

    def __init__(self, cfg: OPTConfig, weights: Dict[str, torch.Tensor], num_layers: Optional[int] = None,
                 fused_norm: bool = True, **attn_kw) -> None:
        self.cfg, self.w, self.fused_norm = cfg, weights, fused_norm
        n = cfg.num_hidden_layers if num_layers is None else num_layers
        self.layers = [HybridOPTDecoderLayer(cfg, weights, f"layers.{i}.", **attn_kw) for i in range(n)]

    def forward(self, input_ids, positions, kv_caches: List[torch.Tensor], shared_cache,
                md: HybridAttentionMetadata) -> torch.Tensor:
        w = self.w
        hidden_states = F.embedding(input_ids, w["embed_tokens"]) + F.embedding(positions + 2, w["embed_positions"])
        if not self.fused_norm or not self.layers:
            for layer, kv in zip(self.layers, kv_caches):
                hidden_states = layer(hidden_states, kv, shared_cache, md)
            return F.layer_norm(hidden_states, (self.cfg.hidden_size,), w["final_ln_w"], w["final_ln_b"])
        normed, _ = ops.add_layer_norm(hidden_states, None, w["layers.0.attn_ln_w"], w["layers.0.attn_ln_b"])
        for i, (layer, kv) in enumerate(zip(self.layers, kv_caches)):
            nxt = f"layers.{i + 1}.attn_ln_" if i + 1 < len(self.layers) else "final_ln_"
            hidden_states, normed = layer.forward_fused_norm(hidden_states, normed, kv, shared_cache, md,
                                                             w[nxt + "w"], w[nxt + "b"])
        return normed

    __call__ = forward

    def next_tokens(self, hidden_states, md: HybridAttentionMetadata) -> torch.Tensor:
        """Greedy next token of every sequence (last row of each prompt / every decode row)."""
        if md.num_prefills:
            last = md.seq_start_loc[1:md.num_prefills + 1].long() - 1
            hidden_states = hidden_states[last]
        logits = hidden_states @ self.w["embed_tokens"].t()
        return logits.argmax(-1)
