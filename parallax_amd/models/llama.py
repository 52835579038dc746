"""Llama-family decoder (covers LlamaForCausalLM and Qwen2ForCausalLM — the
flagship DeepSeek-R1-Distill-Llama-8B is this architecture).

Fresh MI355X-first design (reference analogue: src/parallax/models/llama.py /
qwen2.py): RMSNorm / fused-add-RMSNorm, RoPE, KV scatter, paged attention and
SwiGLU all route through parallax_amd.ops (HIP kernels on GPU); QKV and gate/up
are fused single GEMMs (hipBLASLt); TP via column/row-parallel layers with RCCL
all-reduce over xGMI.
"""

from __future__ import annotations

import math
from typing import Optional

import torch
import torch.nn as nn

from .. import ops
from ..parallel.comm import get_comm
from ..parallel.layers import (
    ColumnParallelLinear,
    MergedColumnParallelLinear,
    RowParallelLinear,
    VocabEmbedding,
    plain_call,
)
from .config import ModelConfig
from .forward_meta import ForwardMeta
from .registry import register_model
from .rope import build_rope_cache_for


class RMSNorm(nn.Module):
    def __init__(self, hidden_size: int, eps: float):
        super().__init__()
        self.weight = nn.Parameter(torch.empty(hidden_size), requires_grad=False)
        self.eps = eps

    def forward(self, x: torch.Tensor, residual: Optional[torch.Tensor] = None):
        if residual is None:
            return ops.rmsnorm(x, self.weight, self.eps)
        return ops.fused_add_rmsnorm(x, residual, self.weight, self.eps)


def norm_project(norm: nn.Module, proj: nn.Module, x: torch.Tensor,
                 residual: Optional[torch.Tensor], gated: bool = False):
    """(proj(norm(x, residual)), the residual then) of a few rows in one launch, gated:
    silu of its first part times the second. None where there is no kernel for it, for
    rows apart and parts that the launches themselves refuse at any number of rows, and
    for modules that are more than these two: hooks and forwards of others see the normed
    rows, which one launch never stores."""
    if x.shape[0] > ops.NORM_LINEAR_MAX_M or not (
            plain_call(norm, RMSNorm.forward)
            and plain_call(proj, MergedColumnParallelLinear.forward)) or proj.fp8 or (
            gated and proj.weight.shape[0] % 16) or (
            residual is not None and not (x.is_contiguous() and residual.is_contiguous())):
        return None
    return ops.norm_linear(x, residual, norm.weight, norm.eps, proj.weight, proj.bias,
                           gated)


def project_norm_mlp(proj: nn.Module, y: torch.Tensor, residual: torch.Tensor,
                     norm: nn.Module, mlp: nn.Module, opens: bool = False):
    """(mlp(norm(proj(y), residual)), the residual then), the projection's parts added
    up by the norm's launch, which also finds the scale of an fp8 MLP's input; opens: of
    the MLP what open_rows() gives. None where there is no kernel for it, for a residual
    of rows apart, which the norm refuses, and for modules that are more than these."""
    if not (parts_of(proj, y.shape[0]) and plain_call(norm, RMSNorm.forward)
            and residual.is_contiguous()):
        return None
    quantize = mlp_takes_fp8(mlp)
    fused = proj.then_norm(y, residual, norm.weight, norm.eps, quantize)
    if fused is None:
        return None
    x, scale, residual = fused
    if opens:
        return mlp.open_rows(x, scale), residual
    return (mlp.from_fp8(x, scale) if quantize else mlp(x)), residual


def runs_as_written(layer: nn.Module) -> bool:
    """Whether calling the layer is its run(), whose result nothing else sees."""
    forward = type(layer).forward
    return getattr(forward, "is_run", False) and plain_call(layer, forward)


def opens_mlp(layer: nn.Module, rows: int) -> bool:
    """Whether the launch behind the layer can add up its MLP's last product."""
    down = getattr(layer.mlp, "down_proj", None)
    return plain_call(layer.mlp, LlamaMLP.forward) and parts_of(
        down, rows) and down.product_alone()


def parts_of(proj: nn.Module, rows: int) -> bool:
    """Whether the projection of that many rows is a product with parts."""
    return isinstance(proj, RowParallelLinear) and ops.product_has_parts(
        rows, proj.weight_fp8 if proj.fp8 else proj.weight)


def mlp_takes_fp8(mlp: nn.Module) -> bool:
    return plain_call(mlp, LlamaMLP.forward) and all(
        plain_call(p, type_.forward) and p.fp8
        for p, type_ in ((mlp.gate_up_proj, MergedColumnParallelLinear),
                         (mlp.down_proj, RowParallelLinear)))


class ResidualLayerNorm(nn.Module):
    """Layer norm (weight and bias) over an fp32 residual stream, fused with
    the scaled update that precedes it: resid += mult * scale * y, then
    (resid - mean) / sqrt(var + eps) * weight + bias in the activation dtype.
    For pre-norm stacks that keep the residual in fp32 and scale each branch
    (layer scale, residual multiplier)."""

    def __init__(self, hidden_size: int, eps: float):
        super().__init__()
        self.weight = nn.Parameter(torch.empty(hidden_size), requires_grad=False)
        self.bias = nn.Parameter(torch.empty(hidden_size), requires_grad=False)
        self.eps = eps

    def forward(self, resid: torch.Tensor, y: Optional[torch.Tensor] = None,
                scale: Optional[torch.Tensor] = None, mult: float = 1.0):
        return ops.add_layernorm(resid, y, scale, mult, self.weight, self.bias,
                                 self.eps, self.weight.dtype)


class LlamaAttention(nn.Module):
    def __init__(self, cfg: ModelConfig, layer_idx: int, local_layer_idx: int):
        super().__init__()
        comm = get_comm()
        self.layer_idx = layer_idx
        self.local_layer_idx = local_layer_idx
        self.head_dim = cfg.head_dim
        self.num_heads = cfg.num_heads // comm.tp_size
        self.num_kv_heads = max(1, cfg.num_kv_heads // comm.tp_size)
        self.scale = self.head_dim ** -0.5
        self.sliding_window = (
            cfg.sliding_window if cfg.layer_type(layer_idx) == "sliding_attention" else -1
        )
        self.qk_norm = cfg.qk_norm
        h = cfg.hidden_size
        self.qkv_proj = MergedColumnParallelLinear(
            h,
            [cfg.num_heads * cfg.head_dim, cfg.num_kv_heads * cfg.head_dim,
             cfg.num_kv_heads * cfg.head_dim],
            bias=cfg.attention_bias,
        )
        self.o_proj = RowParallelLinear(
            cfg.num_heads * cfg.head_dim, h, bias=cfg.o_proj_bias
        )
        self.qk_norm_full = cfg.qk_norm_full
        if self.qk_norm:
            if self.qk_norm_full:
                # minimax-m2: one RMSNorm over the whole concatenated q (and k)
                # width — couples heads, so TP sharding would change the math
                assert comm.tp_size == 1, "full-width qk_norm incompatible with TP"
                self.q_norm = RMSNorm(cfg.num_heads * cfg.head_dim, cfg.rms_norm_eps)
                self.k_norm = RMSNorm(cfg.num_kv_heads * cfg.head_dim, cfg.rms_norm_eps)
            else:
                self.q_norm = RMSNorm(cfg.head_dim, cfg.rms_norm_eps)
                self.k_norm = RMSNorm(cfg.head_dim, cfg.rms_norm_eps)
        self.sinks: Optional[nn.Parameter] = None
        if cfg.attention_sinks:
            self.sinks = nn.Parameter(
                torch.empty(self.num_heads, dtype=torch.float32), requires_grad=False
            )

    def forward(self, x: torch.Tensor, meta: ForwardMeta, rope_cache: torch.Tensor):
        return self.attend(self.qkv_proj(x), x, meta, rope_cache)

    def attend(self, qkv: torch.Tensor, x: torch.Tensor, meta: ForwardMeta,
               rope_cache: torch.Tensor, project: bool = True):
        """The layer from its projection on, to its output projection or before it; x
        only to be handed on."""
        T = qkv.shape[0]
        q, k, v = self.qkv_proj.split_output(qkv)
        # strided views into the fused QKV buffer — no contiguous copies; the
        # HIP kernels take a row stride
        q = q.view(T, self.num_heads, self.head_dim)
        k = k.view(T, self.num_kv_heads, self.head_dim)
        v = v.view(T, self.num_kv_heads, self.head_dim)
        if self.qk_norm:
            if self.qk_norm_full:
                q = self.q_norm(q.reshape(T, -1)).view(T, self.num_heads, self.head_dim)
                k = self.k_norm(k.reshape(T, -1)).view(T, self.num_kv_heads, self.head_dim)
            else:
                q = self.q_norm(q.contiguous())
                k = self.k_norm(k.contiguous())
            v = v.contiguous()
        k_cache, v_cache = meta.kv_cache.layer(self.local_layer_idx)
        sinks = self.sinks.float() if self.sinks is not None else None
        if meta.appends:
            attn = ops.rope_cache_attention_decode(
                q, k, v, k_cache, v_cache, meta.positions, rope_cache,
                meta.slot_mapping, meta.block_tables, meta.seq_lens, self.scale,
                self.sliding_window, sinks=sinks, max_seq_len=meta.max_seq_len or None,
            )
            if attn is not None:
                return self._project_out(attn, x, T) if project else attn.reshape(
                    T, self.num_heads * self.head_dim)
        ops.rope_and_cache(
            q, k, v, k_cache, v_cache, meta.positions, rope_cache,
            meta.slot_mapping,
        )

        if meta.is_prefill:
            attn = ops.prefill_attention(
                q, k_cache, v_cache, meta.block_tables, meta.seq_lens,
                meta.query_lens, self.scale, self.sliding_window, sinks=sinks,
            )
        else:
            attn = ops.paged_attention_decode(
                q, k_cache, v_cache, meta.block_tables, meta.seq_lens,
                self.scale, self.sliding_window, sinks=sinks,
                max_seq_len=meta.max_seq_len or None,
            )
        return self._project_out(attn, x, T) if project else attn.reshape(
            T, self.num_heads * self.head_dim)

    def _project_out(self, attn: torch.Tensor, x: torch.Tensor, T: int):
        """Output projection; subclasses may gate `attn` first (step3p5)."""
        return self.o_proj(attn.reshape(T, self.num_heads * self.head_dim))


class LlamaMLP(nn.Module):
    def __init__(self, cfg: ModelConfig, intermediate_size: Optional[int] = None):
        super().__init__()
        inter = intermediate_size or cfg.intermediate_size
        self.gate_up_proj = MergedColumnParallelLinear(
            cfg.hidden_size, [inter, inter], bias=cfg.mlp_bias
        )
        self.down_proj = RowParallelLinear(inter, cfg.hidden_size, bias=cfg.mlp_bias)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        proj = self.gate_up_proj
        fused = getattr(proj, "silu_and_mul", None)  # another module may stand there
        return self.down_proj(fused(x) if fused else ops.silu_and_mul(proj(x)))

    def open_rows(self, x: torch.Tensor, scale: Optional[torch.Tensor] = None):
        """forward() up to its last product: (rows, their scale or None). scale: x is fp8
        values with it."""
        proj = self.gate_up_proj
        if scale is not None:
            return ops.silu_and_mul_fp8(proj._linear(x, scale))
        fused = getattr(proj, "silu_and_mul", None)
        return fused(x) if fused else ops.silu_and_mul(proj(x)), None

    def from_fp8(self, x: torch.Tensor, scale: torch.Tensor) -> torch.Tensor:
        """forward() of rows that are fp8 values with one scale, by fp8 weights."""
        return self.down_proj.from_fp8(
            *ops.silu_and_mul_fp8(self.gate_up_proj._linear(x, scale)))


class LlamaDecoderLayer(nn.Module):
    def __init__(self, cfg: ModelConfig, layer_idx: int, local_layer_idx: int):
        super().__init__()
        self.self_attn = LlamaAttention(cfg, layer_idx, local_layer_idx)
        self.mlp = LlamaMLP(cfg)
        self.input_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
        self.post_attention_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)

    def forward(self, x, residual, meta: ForwardMeta, rope_cache):
        return self.run(x, residual, meta, rope_cache)

    forward.is_run = True

    def run(self, x, residual, meta: ForwardMeta, rope_cache, normed: bool = False,
            opens: bool = False):
        """normed: x is the input norm's result and residual what it added up. opens: of
        the MLP what open_rows() gives, in place of its result."""
        # sizes first: a prompt's layers wait for the host
        rows = x.shape[0]
        if not (normed or opens) and (
                rows > ops.SKINNY_GEMM_MAX_M or rows > ops.NORM_LINEAR_MAX_M
                and not parts_of(getattr(self.self_attn, "o_proj", None), rows)):
            if residual is None:
                residual = x
                x = self.input_layernorm(x)
            else:
                x, residual = self.input_layernorm(x, residual)
            x = self.self_attn(x, meta, rope_cache)
            x, residual = self.post_attention_layernorm(x, residual)
            return self.mlp(x), residual
        attn, mlp = self.self_attn, self.mlp
        fused = None
        plain = plain_call(attn, LlamaAttention.forward) and (
            type(attn)._project_out is LlamaAttention._project_out)
        if plain and not normed:
            fused = norm_project(self.input_layernorm, attn.qkv_proj, x, residual)
        if fused is not None:
            qkv, residual = fused
        else:
            if not normed:
                x, residual = self._input_norm(x, residual)
            qkv = attn.qkv_proj(x) if plain else None
        if plain:
            y = attn.attend(qkv, x, meta, rope_cache, project=False)
            fused = project_norm_mlp(attn.o_proj, y, residual,
                                     self.post_attention_layernorm, mlp, opens)
            if fused is not None:
                return fused
            x = attn.o_proj(y)
        else:
            x = attn(x, meta, rope_cache)
        if not opens and plain_call(mlp, LlamaMLP.forward):
            fused = norm_project(self.post_attention_layernorm, mlp.gate_up_proj, x,
                                 residual, gated=True)
            if fused is not None:
                x, residual = fused
                return mlp.down_proj(x), residual
        x, residual = self.post_attention_layernorm(x, residual)
        return (mlp.open_rows(x) if opens else mlp(x)), residual

    def _input_norm(self, x, residual):
        if residual is None:
            return self.input_layernorm(x), x
        return self.input_layernorm(x, residual)


def stack_in_one(layers, hidden: torch.Tensor, meta: ForwardMeta,
                 rope_cache: torch.Tensor):
    """What the layers make of a decode step of a few rows, in one launch: (the last
    one's branch, the residual stream). None where there is no kernel for it and for
    layers that are more than LlamaDecoderLayer, of one width, without windows, sinks,
    norms of heads and quantised weights."""
    if not (meta.appends and meta.max_seq_len and hidden.is_cuda and layers) or (
            hidden.dim() != 2 or hidden.shape[0] > ops.NORM_LINEAR_MAX_M
            or not plain_call(layers[0], LlamaDecoderLayer.forward)):
        return None
    a0, norm = layers[0].self_attn, layers[0].input_layernorm
    if not (plain_call(a0, LlamaAttention.forward)
            and plain_call(layers[0].mlp, LlamaMLP.forward)
            and plain_call(norm, RMSNorm.forward)) or not ops.decode_stack_has(
            *hidden.shape, a0.num_heads, a0.num_kv_heads, a0.head_dim,
            getattr(layers[0].mlp.down_proj, "in_per_rank", 0), meta.max_seq_len):
        return None
    # what an eager step can be refused for as a whole, before its layers are looked at
    k_cache = meta.kv_cache.layer(a0.local_layer_idx)[0]
    if not hidden.dtype == k_cache.dtype == torch.bfloat16 or (
            rope_cache.shape[-1] != a0.head_dim
            or torch.is_grad_enabled() and hidden.requires_grad):
        return None
    eps = norm.eps
    tensors = []
    for layer in layers:
        if not plain_call(layer, LlamaDecoderLayer.forward):
            return None
        attn, mlp = layer.self_attn, layer.mlp
        if not (plain_call(attn, LlamaAttention.forward)
                and getattr(attn.attend, "__func__", None) is LlamaAttention.attend
                and getattr(attn._project_out, "__func__", None)
                is LlamaAttention._project_out
                and plain_call(mlp, LlamaMLP.forward)):
            return None
        norms = layer.input_layernorm, layer.post_attention_layernorm
        up, down = (attn.qkv_proj, mlp.gate_up_proj), (attn.o_proj, mlp.down_proj)
        if not (all(plain_call(n, RMSNorm.forward) and n.eps == eps for n in norms)
                and all(plain_call(p, MergedColumnParallelLinear.forward)
                        and not p.fp8 for p in up)
                and all(plain_call(p, RowParallelLinear.forward) and not p.fp8
                        and p.tp_size == 1 and p.bias is None for p in down)):
            return None
        if attn.qk_norm or attn.sinks is not None or attn.sliding_window > 0 or (
                up[1].bias is not None or attn.scale != a0.scale
                or (attn.num_heads, attn.num_kv_heads) != (a0.num_heads, a0.num_kv_heads)):
            return None
        w_qkv, b_qkv = up[0].weight, up[0].bias
        tensors += [norms[0].weight, w_qkv,
                    w_qkv.new_empty(0) if b_qkv is None else b_qkv, down[0].weight,
                    norms[1].weight, up[1].weight, down[1].weight,
                    *meta.kv_cache.layer(attn.local_layer_idx)]
    return ops.decode_stack(
        hidden, tensors, eps, a0.num_heads, a0.num_kv_heads, a0.scale,
        meta.positions, rope_cache, meta.slot_mapping, meta.block_tables, meta.seq_lens,
        meta.max_seq_len)


@register_model("LlamaForCausalLM", "Qwen2ForCausalLM", "MistralForCausalLM")
class LlamaShardModel(nn.Module):
    """A contiguous layer range [start_layer, end_layer) of a Llama-family model.
    First shard owns the embedding; last shard owns final norm + lm_head
    (reference base_executor.py:124-125 stage-role convention)."""

    decoder_layer_cls = LlamaDecoderLayer

    def __init__(self, cfg: ModelConfig, start_layer: int = 0, end_layer: Optional[int] = None):
        super().__init__()
        self.cfg = cfg
        self.start_layer = start_layer
        self.end_layer = end_layer if end_layer is not None else cfg.num_layers
        self.is_first = start_layer == 0
        self.is_last = self.end_layer == cfg.num_layers

        if self.is_first:
            self.embed_tokens = VocabEmbedding(cfg.vocab_size, cfg.hidden_size)
        self.layers = nn.ModuleList(
            self._build_layers(cfg, start_layer, self.end_layer)
        )
        if self.is_last:
            self.norm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
            self.lm_head = ColumnParallelLinear(cfg.hidden_size, cfg.vocab_size,
                                                gather_output=True)
        self.register_buffer(
            "rope_cache",
            build_rope_cache_for(cfg, rot_dim=cfg.rot_dim),
            persistent=False,
        )

    def _build_layers(self, cfg: ModelConfig, start: int, end: int):
        return [
            self.decoder_layer_cls(cfg, g, i)
            for i, g in enumerate(range(start, end))
        ]

    @property
    def num_local_layers(self) -> int:
        return len(self.layers)

    def embed(self, input_ids: torch.Tensor) -> torch.Tensor:
        assert self.is_first, "only the first shard embeds tokens"
        return self.embed_tokens(input_ids)

    def forward(self, hidden: torch.Tensor, meta: ForwardMeta) -> torch.Tensor:
        """hidden: [T, hidden] — embeddings on the first shard, the previous
        stage's output elsewhere. Returns [T, hidden] post final-norm on the
        last shard, pre-norm activations otherwise."""
        residual = None
        fused = stack_in_one(self.layers, hidden, meta, self.rope_cache)
        if fused is not None:
            hidden, residual = fused
        elif hidden.dim() == 2 and (
                ops.NORM_LINEAR_MAX_M < hidden.shape[0] <= ops.SKINNY_GEMM_MAX_M):
            hidden, residual, done = self._few_rows(hidden, meta)
            if done:
                return hidden
        else:
            for layer in self.layers:
                hidden, residual = layer(hidden, residual, meta, self.rope_cache)
        if self.is_last:
            if residual is None:  # post-norm families (minimax) fold residuals
                hidden = self.norm(hidden)
            else:
                hidden, _ = self.norm(hidden, residual)
        elif residual is not None:
            hidden = hidden + residual
        return hidden

    def _few_rows(self, hidden: torch.Tensor, meta: ForwardMeta):
        """The layers of a few rows: (hidden, residual, whether hidden is what the forward
        returns). The parts of an MLP's last product are added up by the launch of the
        norm that follows, or of the sum behind the last layer, where both modules are
        what they are here and nothing looks on."""
        rows, residual, normed = hidden.shape[0], None, False
        runs = [hidden.is_cuda and runs_as_written(x) for x in self.layers]
        for i, layer in enumerate(self.layers):
            last = i + 1 == len(self.layers)
            if last:
                norm = self.norm if self.is_last else None
            else:
                norm = self.layers[i + 1].input_layernorm if runs[i + 1] else None
            follows = last and not self.is_last or (
                norm is not None and plain_call(norm, RMSNorm.forward))
            opens = runs[i] and follows and opens_mlp(layer, rows)
            if not (normed or opens):
                hidden, residual = layer(hidden, residual, meta, self.rope_cache)
                continue
            hidden, residual = layer.run(hidden, residual, meta, self.rope_cache, normed,
                                         opens)
            normed = False
            if not opens:
                continue
            (rows_in, scale), down = hidden, layer.mlp.down_proj
            weight = down.weight_fp8 if down.fp8 else down.weight
            w_scale = down.weight_scale if down.fp8 else None
            if norm is not None:
                fused = ops.linear_norm(rows_in, weight, w_scale, residual, norm.weight,
                                        norm.eps, x_scale=scale)
                if fused is not None:
                    hidden, residual, normed = fused[0], fused[2], True
            else:
                fused = ops.linear_add(rows_in, weight, w_scale, residual, x_scale=scale)
                if fused is not None:
                    hidden, normed = fused, True
            if fused is None:
                hidden = down(rows_in) if scale is None else down.from_fp8(rows_in, scale)
        return hidden, residual, normed

    def compute_logits(self, hidden: torch.Tensor) -> torch.Tensor:
        assert self.is_last, "only the last shard computes logits"
        # lm_head is a ColumnParallelLinear (gathers under TP) and already
        # routes through ops.linear -> the tuned hipBLASLt path
        return self.lm_head(
            hidden.to(self.lm_head.weight.dtype).contiguous()
        ).float()

    # -- weight loading ---------------------------------------------------------

    _STACKED = {
        "q_proj": ("qkv_proj", 0),
        "k_proj": ("qkv_proj", 1),
        "v_proj": ("qkv_proj", 2),
        "gate_proj": ("gate_up_proj", 0),
        "up_proj": ("gate_up_proj", 1),
    }

    def map_global_layer(self, name: str) -> Optional[str]:
        """'model.layers.<g>.rest' -> 'layers.<local>.rest' (None if out of range);
        parity with the reference shard loader's key remap (shard_loader.py:229)."""
        if name.startswith("model.layers."):
            parts = name.split(".")
            g = int(parts[2])
            if not (self.start_layer <= g < self.end_layer):
                return None
            return ".".join(["layers", str(g - self.start_layer)] + parts[3:])
        if name.startswith("model.embed_tokens."):
            if self.is_first:
                return name.replace("model.", "", 1)
            if self.is_last and self.cfg.tie_word_embeddings:
                return name.replace("model.embed_tokens", "lm_head")
            return None
        if name.startswith("model.norm."):
            return name.replace("model.", "", 1) if self.is_last else None
        if name.startswith("lm_head."):
            return name if self.is_last and not self.cfg.tie_word_embeddings else None
        return None

    def load_hf_weight(self, name: str, tensor: torch.Tensor) -> bool:
        """Route one HF-named tensor into this shard. Returns True if consumed."""
        local = self.map_global_layer(name)
        if local is None:
            return False
        parts = local.split(".")
        leaf = parts[-1]  # 'weight' or 'bias'
        stem = parts[-2]
        tensor = tensor.to(torch.bfloat16)
        if stem in self._STACKED:
            target_name, idx = self._STACKED[stem]
            module = self._resolve(parts[:-2] + [target_name])
            module.load_full_weight_part(idx, tensor if leaf == "weight" else None,
                                         tensor if leaf == "bias" else None)
            return True
        module = self._resolve(parts[:-1])
        if isinstance(module, (ColumnParallelLinear, RowParallelLinear)):
            module.load_full_weight(tensor if leaf == "weight" else None,
                                    tensor if leaf == "bias" else None)
        else:
            getattr(module, leaf).data.copy_(tensor)
        return True

    def _resolve(self, path_parts):
        mod = self
        for p in path_parts:
            mod = mod[int(p)] if p.isdigit() else getattr(mod, p)
        return mod

    @torch.no_grad()
    def init_random(self, seed: int = 1234) -> None:
        """Random-init all parameters (synthetic-weight benchmarking; no network
        for checkpoints). Norm weights -> 1, linears -> N(0, 0.02/sqrt(2L))."""
        g = torch.Generator().manual_seed(seed)
        std = 0.02 / math.sqrt(2 * max(1, self.cfg.num_layers))
        for name, p in self.named_parameters():
            if "norm" in name.lower():
                p.data.fill_(1.0)
            elif name.endswith("bias"):
                p.data.zero_()
            elif "embed" in name or "lm_head" in name:
                p.data.copy_(
                    torch.randn(p.shape, generator=g, dtype=torch.float32).mul_(0.02)
                    .to(p.dtype)
                )
            else:
                p.data.copy_(
                    torch.randn(p.shape, generator=g, dtype=torch.float32).mul_(std)
                    .to(p.dtype)
                )


