"""Dense Qwen3 language model around the drop-in attention (model/transformer.py:24-162).

A mirror of the reference's ``Qwen3Model`` / ``TransformerBlock`` with the same
submodule names, so the reference's state dicts load unchanged:
``embed.embed_tokens``, ``layers.{i}.input_layernorm``, ``layers.{i}.attention``
(the drop-in ``Attention``), ``layers.{i}.post_attention_layernorm``,
``layers.{i}.feed_forward.{gate,up,down}_proj``, ``norm``, ``lm_head``.  The
forward signature and the returned dict are the reference's
(transformer.py:107-156).

Attention, the layer RMSNorms and SwiGLU's product run on the gfx950 kernels (the
latter two as tensor operations where ``ops.plain_rows`` says no: host tensors,
other dtypes, transforms); embedding, the projections and the LM head are the
reference's torch ops (hipBLASLt GEMMs).  MoE
layers (model/moe.py) are outside the attention hot path and not provided.
``gradient_checkpointing`` (config field and attribute, transformer.py:92,
121-127) recomputes each block in the backward when training, as the
reference does.
"""

from __future__ import annotations

from dataclasses import dataclass
from typing import List, Optional

import torch
import torch.nn as nn
import torch.nn.functional as F
import torch.utils.checkpoint as checkpoint_utils

from . import _lib, ops
from .attention import Attention, KVCache
from .config import AttentionConfig
from .norm import LayerRMSNormFn, layer_rms_norm, plain_rms_norm


@dataclass
class ModelConfig(AttentionConfig):
    """The dense-model fields of model/config.py:14-83 on top of the attention ones."""

    vocab_size: int = 151936
    num_hidden_layers: int = 32
    intermediate_size: int = 11008
    tie_word_embeddings: bool = False
    initializer_range: float = 0.02
    gradient_checkpointing: bool = False


class LayerRMSNorm(nn.Module):
    """RMSNorm over the hidden size, the reference's arithmetic (model/norm.py:17-22):
    fp32 statistic, cast back to the input dtype before the weight multiply.

    Under autograd a bf16 input is copied, so that its owner may write to it before the
    backward (the tensor operations keep an fp32 copy; of an fp32 input they keep the input
    itself, and so does this).  The model's own norms do too: a program may call them by
    themselves, and hooks see their inputs.  ``input_kept`` says that nobody writes to the
    input until then, and autograd keeps the input itself."""

    input_kept = False  # of a module that was pickled without it

    def __init__(self, hidden_size: int, eps: float = 1e-6, input_kept: bool = False):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(hidden_size))
        self.eps = eps
        self.input_kept = input_kept

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        w = self.weight
        # as tensor operations eight launches forward and some twenty backward, each a
        # pass over fp32 rows: a training block at 4096 x 2048 bf16, with SwiGLU's
        # product below, 2296 -> 1863 us, and 9 for each copy; four layers on 173 tokens
        # 1420 -> 1286 us
        if not torch.jit.is_scripting():
            grad = ops.takes_gradient(x, w)
            if (grad is not None and w.dim() == 1 and not (grad and w.shape[0] > 4096)
                    and x.shape[-1:] == w.shape and ops.plain_rows(x, w)):
                if not grad:
                    return plain_rms_norm(x, w, self.eps)
                kept = self.input_kept or x.dtype == torch.float32
                return LayerRMSNormFn.apply(x if kept else x.clone(), w, self.eps)
        return layer_rms_norm(x, w, self.eps)


def _swiglu_product(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    y = torch.empty_like(gate)
    rc = _lib.load().nq_swiglu(ops._ptr(gate), ops._ptr(up), ops._ptr(y), gate.numel(), ops._code(gate),
                               ops._stream(gate))
    _lib.check(rc, "nq_swiglu")
    return y


# Elements of gate from which a product with a gradient goes through the kernels.  An
# autograd function's calls take the host ~35 us longer than the tensor operations' (2048
# rows of 1024 -> 3072, forward and backward: 344 us against 309); from here on the
# device takes longer than the host, and its passes count (4096 rows: 351 against 375).
_SWIGLU_GRAD_ELEMENTS = 1 << 23


class _SwiGLUProduct(torch.autograd.Function):
    """silu(gate) * up on the kernels; for tensors that ``ops.plain_rows`` accepts."""

    @staticmethod
    def forward(ctx, gate, up):
        ctx.save_for_backward(gate, up)
        return _swiglu_product(gate, up)

    @staticmethod
    def backward(ctx, dy):
        gate, up = ctx.saved_tensors
        dyc = dy.contiguous()
        if torch.is_grad_enabled() or not ops.plain_rows(gate, up, dyc):
            # a gradient of the gradient, or one under a transform: tensor operations
            s = torch.sigmoid(gate.float())
            dg = (dy * up).float() * s * (1 + gate.float() * (1 - s))
            return dg.to(gate.dtype), dy * F.silu(gate)
        dgate, dup = torch.empty_like(gate), torch.empty_like(up)
        rc = _lib.load().nq_swiglu_bwd(ops._ptr(gate), ops._ptr(up), ops._ptr(dyc), ops._ptr(dgate), ops._ptr(dup),
                                       gate.numel(), ops._code(gate), ops._stream(gate))
        _lib.check(rc, "nq_swiglu_bwd")
        return dgate, dup


class SwiGLU(nn.Module):
    """model/ffn.py:17-28: down(silu(gate(x)) * up(x))."""

    def __init__(self, hidden_size: int, intermediate_size: int):
        super().__init__()
        self.gate_proj = nn.Linear(hidden_size, intermediate_size, bias=False)
        self.up_proj = nn.Linear(hidden_size, intermediate_size, bias=False)
        self.down_proj = nn.Linear(intermediate_size, hidden_size, bias=False)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        gate, up = self.gate_proj(x), self.up_proj(x)
        if not torch.jit.is_scripting():
            grad = ops.takes_gradient(gate, up)
            if (grad is not None and not (grad and gate.numel() < _SWIGLU_GRAD_ELEMENTS)
                    and gate.dtype == up.dtype and gate.shape == up.shape and ops.plain_rows(gate, up)):
                return self.down_proj(_SwiGLUProduct.apply(gate, up) if grad else _swiglu_product(gate, up))
        return self.down_proj(F.silu(gate) * up)


class TokenEmbedding(nn.Module):
    """model/embedding.py:9-16."""

    def __init__(self, config):
        super().__init__()
        self.embed_tokens = nn.Embedding(config.vocab_size, config.hidden_size)

    def forward(self, input_ids: torch.Tensor) -> torch.Tensor:
        return self.embed_tokens(input_ids)


def _check_dense(config) -> None:
    if getattr(config, "is_moe", False):
        raise NotImplementedError("MoE layers are outside the attention hot path; dense models only")


class TransformerBlock(nn.Module):
    """Pre-norm block (transformer.py:24-76): x += Attn(norm(x)); x += FFN(norm(x))."""

    def __init__(self, config, layer_idx: int = 0):
        super().__init__()
        _check_dense(config)
        self.layer_idx = layer_idx
        self.config = config
        self.input_layernorm = LayerRMSNorm(config.hidden_size, eps=config.rms_norm_eps)
        self.attention = Attention(config, layer_idx=layer_idx)
        self.post_attention_layernorm = LayerRMSNorm(config.hidden_size, eps=config.rms_norm_eps)
        self.feed_forward = SwiGLU(config.hidden_size, config.intermediate_size)

    def forward(self, hidden_states: torch.Tensor, position_ids: Optional[torch.Tensor] = None,
                attention_mask: Optional[torch.Tensor] = None,
                kv_cache: Optional[KVCache] = None):
        residual = hidden_states
        hidden_states = self.attention(self.input_layernorm(hidden_states), position_ids,
                                       attention_mask, kv_cache)
        hidden_states = residual + hidden_states
        residual = hidden_states
        hidden_states = residual + self.feed_forward(self.post_attention_layernorm(hidden_states))
        return hidden_states, None


class Qwen3Model(nn.Module):
    """Embedding -> blocks -> RMSNorm -> LM head (transformer.py:78-156)."""

    def __init__(self, config):
        super().__init__()
        _check_dense(config)
        self.config = config
        self.embed = TokenEmbedding(config)
        self.layers = nn.ModuleList([TransformerBlock(config, layer_idx=i)
                                     for i in range(config.num_hidden_layers)])
        self.norm = LayerRMSNorm(config.hidden_size, eps=config.rms_norm_eps)
        self.lm_head = nn.Linear(config.hidden_size, config.vocab_size, bias=False)
        if getattr(config, "tie_word_embeddings", False):
            self.lm_head.weight = self.embed.embed_tokens.weight
        # transformer.py:92: each block recomputed in the backward when training
        self.gradient_checkpointing = getattr(config, "gradient_checkpointing", False)
        self.apply(self._init_weights)

    def _init_weights(self, module: nn.Module) -> None:
        std = getattr(self.config, "initializer_range", 0.02)
        if isinstance(module, nn.Linear):
            nn.init.normal_(module.weight, mean=0.0, std=std)
            if module.bias is not None:
                nn.init.zeros_(module.bias)
        elif isinstance(module, nn.Embedding):
            nn.init.normal_(module.weight, mean=0.0, std=std)

    def set_cache_semantics(self, fixed: bool) -> None:
        """``fixed=True``: a prefill into a cache is causal and positions continue
        from the cache length (``Attention.rope_positions = "cache"``,
        ``cache_prefill_causal = True``).  ``False`` keeps the reference's
        behaviour (bidirectional cache prefill, positions from 0)."""
        for layer in self.layers:
            layer.attention.rope_positions = "cache" if fixed else "reference"
            layer.attention.cache_prefill_causal = bool(fixed)

    def forward(self, input_ids: torch.Tensor, position_ids: Optional[torch.Tensor] = None,
                attention_mask: Optional[torch.Tensor] = None,
                kv_caches: Optional[List[KVCache]] = None,
                labels: Optional[torch.Tensor] = None) -> dict:
        hidden_states = self.embed(input_ids)
        for i, layer in enumerate(self.layers):
            kv_cache = kv_caches[i] if kv_caches is not None else None
            if self.gradient_checkpointing and self.training:
                # transformer.py:121-127: the block's activations (the attention
                # kernels' Q-hat, K-hat, O and LSE included) are dropped and the
                # block's forward runs again inside the backward
                hidden_states, _ = checkpoint_utils.checkpoint(
                    layer, hidden_states, position_ids, attention_mask, kv_cache, use_reentrant=False)
            else:
                hidden_states, _ = layer(hidden_states, position_ids, attention_mask, kv_cache)
        hidden_states = self.norm(hidden_states)
        logits = self.lm_head(hidden_states)
        loss = None
        if labels is not None:
            loss = F.cross_entropy(logits[..., :-1, :].contiguous().view(-1, logits.shape[-1]),
                                   labels[..., 1:].contiguous().view(-1), ignore_index=-100)
        return {"logits": logits, "loss": loss, "aux_loss": None, "hidden_states": hidden_states}

    @torch.no_grad()
    def count_parameters(self) -> dict:
        """transformer.py:158-162."""
        total = sum(p.numel() for p in self.parameters())
        trainable = sum(p.numel() for p in self.parameters() if p.requires_grad)
        return {"total": total, "trainable": trainable}
