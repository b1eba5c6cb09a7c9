"""Minimal Llama decoder host that drives the KV data path through its real call sites.

It plays the role of hexgen_core's GPTLMHeadModel for the Llama subset the
pilot runs (pre-norm blocks, RMSNorm, rotary q/k, GQA attention with a KV
cache, SwiGLU MLP, untied LM head; hexgen/hexgen_core/models/gpt.py:363-483,
modules/block.py:112-175, mlp.py:63-87, rms_norm.py:6-15).  Weights are read
in HuggingFace Llama layout from safetensors.  Per layer and step the cache
calls are exactly the reference's: ``_update_kv_cache`` then
``FlashCrossAttention`` (mha.py:565-569), or the fused HIP append+attend;
with ``fused_ft_kernel`` the decode steps call
``_apply_rotary_single_query_attention`` on unrotated q/k (mha.py:553-571).
Dense projections use torch (hipBLASLt), with q/k/v and gate/up each one
product (joined once when the host is built, which takes about 1.3 times as
long for it); the steps between them are one hexkv launch each (residual sum
and RMSNorm, head split and rotary, SwiGLU).  For one or two tokens the
products are hexkv's too (``ops.norm_linear``, ``ops.norm_rope_linear``), with
the norm before and the rotary or SwiGLU after them in the same launch.  Every
KV byte moves through hexkv.
"""
from __future__ import annotations

import json
from dataclasses import dataclass
from pathlib import Path

import torch
import torch.nn.functional as F

from . import ops
from .mha import FlashCrossAttention, _apply_rotary_single_query_attention, _update_kv_cache, update_and_attend


@dataclass
class LlamaShape:
    vocab_size: int
    hidden_size: int
    intermediate_size: int
    num_hidden_layers: int
    num_attention_heads: int
    num_key_value_heads: int
    rms_norm_eps: float = 1e-6
    rope_theta: float = 10000.0
    max_position_embeddings: int = 2048
    tie_word_embeddings: bool = False

    @property
    def head_dim(self) -> int:
        return self.hidden_size // self.num_attention_heads

    @classmethod
    def from_config(cls, config: dict) -> "LlamaShape":
        if config.get("model_type") != "llama" or config.get("rope_scaling") is not None:
            raise ValueError("This baseline supports Llama architecture without RoPE scaling")
        theta = config.get("rope_theta")
        if theta is None:
            theta = (config.get("rope_parameters") or {}).get("rope_theta", 10000.0)
        return cls(vocab_size=config["vocab_size"], hidden_size=config["hidden_size"],
                   intermediate_size=config["intermediate_size"],
                   num_hidden_layers=config["num_hidden_layers"],
                   num_attention_heads=config["num_attention_heads"],
                   num_key_value_heads=config.get("num_key_value_heads") or config["num_attention_heads"],
                   rms_norm_eps=config.get("rms_norm_eps", 1e-6), rope_theta=float(theta),
                   max_position_embeddings=config.get("max_position_embeddings", 2048),
                   tie_word_embeddings=bool(config.get("tie_word_embeddings", False)))


def read_config(model_dir) -> dict:
    return json.loads((Path(model_dir) / "config.json").read_text())


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    """rms_norm.py:13-15: normalise in fp32, cast back, scale: the plain form
    of what ``ops.add_rms_norm`` computes in one launch."""
    normalized = x.float() * torch.rsqrt(x.float().square().mean(-1, keepdim=True) + eps)
    return normalized.to(x.dtype) * weight


class LlamaHost:
    """Greedy-decode host; ``forward`` mirrors GPTLMHeadModel.forward's
    ``(input_ids, inference_params, last_token_only)`` contract."""

    def __init__(self, shape: LlamaShape, weights: dict, device, dtype):
        self.shape = shape
        self.device, self.dtype = torch.device(device), dtype
        w = {k: v.to(device=self.device, dtype=dtype) for k, v in weights.items()}
        self.embed = w["model.embed_tokens.weight"]
        self.norm = w["model.norm.weight"].contiguous()
        self.lm_head = w["model.embed_tokens.weight"] if shape.tie_word_embeddings else w["lm_head.weight"]
        self.layers = []
        for i in range(shape.num_hidden_layers):
            p = f"model.layers.{i}."
            # projections of one input are one matrix each, laid out once
            self.layers.append({
                "ln1": w[p + "input_layernorm.weight"].contiguous(),
                "ln2": w[p + "post_attention_layernorm.weight"].contiguous(),
                "wqkv": torch.cat([w.pop(p + f"self_attn.{n}_proj.weight") for n in "qkv"]),
                "wo": w[p + "self_attn.o_proj.weight"],
                "gate_up": torch.cat([w.pop(p + f"mlp.{n}_proj.weight") for n in ("gate", "up")]),
                "down": w[p + "mlp.down_proj.weight"],
            })
        d = shape.head_dim
        self.inv_freq = 1.0 / (shape.rope_theta ** (torch.arange(0, d, 2, device=self.device,
                                                                  dtype=torch.float32) / d))
        self.scale = d ** -0.5  # gpt.py:72
        self.attn = FlashCrossAttention(causal=True, softmax_scale=self.scale)

    @classmethod
    def load(cls, model_dir, device, dtype) -> "LlamaHost":
        from safetensors.torch import load_file
        shape = LlamaShape.from_config(read_config(model_dir))
        shards = sorted(Path(model_dir).glob("*.safetensors"))
        if not shards:
            raise ValueError("A local safetensors checkpoint is required")
        state = {}
        for shard in shards:
            values = load_file(str(shard), device="cpu")
            if set(state).intersection(values):
                raise ValueError("Duplicate checkpoint keys")
            state.update(values)
        return cls(shape, state, device, dtype)

    def _norm_linear(self, h, y, norm, weight, glu=False, keep_sum=True):
        """``(product, h + y)`` of RMSNorm(h + y) and ``weight``, with ``glu``
        SwiGLU of its two halves: one launch for a few tokens, else the norm's,
        the library product and the SwiGLU's."""
        if ops.linear_fits(h, norm, weight):
            return ops.norm_linear(h, y, norm, self.shape.rms_norm_eps, weight, glu, keep_sum)
        x = F.linear(ops.add_rms_norm(h, y, norm, self.shape.rms_norm_eps, keep_sum), weight)
        return (ops.silu_mul(x) if glu else x), h

    def _linear(self, x, weight):
        if ops.linear_fits(x, weight):
            return ops.norm_linear(x, None, None, 0.0, weight)[0]
        return F.linear(x, weight)

    @torch.inference_mode()
    def forward(self, input_ids: torch.Tensor, inference_params, last_token_only: bool = True,
                fused_append: bool = False) -> torch.Tensor:
        s = self.shape
        batch, seqlen = input_ids.shape
        d = s.head_dim
        offset = inference_params.sequence_len_offset
        # A ragged decode batch: each sequence's token sits at its own cached
        # length (lengths_per_sample, generation.py:30).
        positions = None
        if inference_params.lengths_per_sample is not None and seqlen == 1 and offset > 0:
            b0 = inference_params.batch_size_offset
            positions = inference_params.lengths_per_sample[b0:b0 + batch].to(torch.int32).contiguous()
        heads, kv_heads = s.num_attention_heads, s.num_key_value_heads
        h = F.embedding(input_ids, self.embed)
        y = None  # the block output still to be added to h
        for i, layer in enumerate(self.layers):
            if inference_params.fused_ft_kernel and offset > 0:
                # FT decode (mha.py:553-571): rotary, append and attention in one call
                qkv, h = self._norm_linear(h, y, layer["ln1"], layer["wqkv"])
                q = qkv[..., :heads * d].view(batch, seqlen, heads, d)
                kv = qkv[..., heads * d:].view(batch, seqlen, 2, kv_heads, d)
                context = _apply_rotary_single_query_attention(q, inference_params, i, d, s.rope_theta, kv=kv)
            else:
                if ops.linear_fits(h, layer["ln1"], layer["wqkv"]):
                    q, kv, h = ops.norm_rope_linear(h, y, layer["ln1"], s.rms_norm_eps, layer["wqkv"], heads, kv_heads, d,
                                                    self.inv_freq, offset, positions)
                else:
                    qkv, h = self._norm_linear(h, y, layer["ln1"], layer["wqkv"])
                    q, kv = ops.rope_split(qkv, heads, kv_heads, d, self.inv_freq, offset, positions)
                if fused_append and offset > 0 and seqlen == 1 and i in inference_params.key_value_memory_dict:
                    context = update_and_attend(q, kv, inference_params, i, self.scale)
                else:
                    kv_view = _update_kv_cache(kv, inference_params, i)
                    # prompt (offset 0): causal; decode: causal=False (mha.py:566-569)
                    context = self.attn(q, kv_view, causal=None if offset == 0 else False)
            y = self._linear(context.reshape(batch, seqlen, -1), layer["wo"])
            x, h = self._norm_linear(h, y, layer["ln2"], layer["gate_up"], glu=True)
            y = self._linear(x, layer["down"])
        if last_token_only:
            h, y = h[:, -1], None if y is None else y[:, -1]
        return self._norm_linear(h, y, self.norm, self.lm_head, keep_sum=False)[0]
