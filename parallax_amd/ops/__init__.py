"""Op dispatch: hand-written HIP/CDNA4 kernels on GPU, eager torch on CPU.

Policy (per the MI355X-first design): on a CUDA (= ROCm/HIP) device the compiled
extension `parallax_amd._C` is REQUIRED for the core hot ops — if it is missing
the op raises instead of silently falling back to eager torch, so a GPU run can
never "pass" on a Python fallback. On CPU the fp32 reference implementations run
(plumbing tests, no GPU in CI).
"""

from __future__ import annotations

import os
from typing import List, Optional, Sequence, Tuple

import torch

from . import reference as ref
from ..utils.logging_config import get_logger

logger = get_logger("ops")

_EXT = None
_EXT_ERR: Optional[str] = None
_warned_prefill = False


def _try_load_extension():
    global _EXT, _EXT_ERR
    if _EXT is not None or _EXT_ERR is not None:
        return _EXT
    try:
        from . import _C  # built in-tree by setup.py build_ext --inplace

        _EXT = _C
        logger.info("loaded HIP extension parallax_amd.ops._C")
    except ImportError as e:  # pragma: no cover - exercised only without build
        _EXT_ERR = str(e)
    return _EXT


def has_extension() -> bool:
    return _try_load_extension() is not None


def _require_ext(op_name: str):
    ext = _try_load_extension()
    if ext is None:
        raise RuntimeError(
            f"parallax_amd HIP extension is required for {op_name} on GPU but is not "
            f"built (import error: {_EXT_ERR}). Build it with "
            f"`python setup.py build_ext --inplace` (PYTORCH_ROCM_ARCH=gfx950)."
        )
    return ext


# -- normalization ------------------------------------------------------------


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-6) -> torch.Tensor:
    if x.is_cuda:
        ext = _require_ext("rmsnorm")
        out = torch.empty_like(x)
        ext.rmsnorm(out, x.contiguous(), weight, eps)
        return out
    return ref.rmsnorm(x, weight, eps)


def fused_add_rmsnorm(
    x: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, eps: float = 1e-6
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Returns (normed, new_residual). On GPU this mutates x (normed) and
    residual (sum) in place to avoid two extra HBM round trips."""
    if x.is_cuda:
        ext = _require_ext("fused_add_rmsnorm")
        ext.fused_add_rmsnorm(x, residual, weight, eps)
        return x, residual
    return ref.fused_add_rmsnorm(x, residual, weight, eps)


# -- rotary -------------------------------------------------------------------

build_rope_cache = ref.build_rope_cache


def rope_inplace(
    q: torch.Tensor,
    k: Optional[torch.Tensor],
    positions: torch.Tensor,
    cos_sin: torch.Tensor,
    is_neox: bool = True,
) -> None:
    if q.is_cuda:
        ext = _require_ext("rope")
        ext.rope_inplace(
            q,
            k if k is not None else q[:0],
            positions.to(torch.int32),
            cos_sin,
            is_neox,
        )
        return
    ref.rope_inplace(q, k, positions, cos_sin, is_neox)


# -- cache scatter ---------------------------------------------------------------


def rope_and_cache(
    q: torch.Tensor,             # [T, Hq, D] (rows may be strided, e.g. QKV views)
    k: torch.Tensor,             # [T, Hk, D]
    v: torch.Tensor,             # [T, Hk, D]
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    positions: torch.Tensor,
    cos_sin: torch.Tensor,
    slot_mapping: torch.Tensor,
    is_neox: bool = True,
    k_scale: float = 1.0,
    v_scale: float = 1.0,
) -> None:
    """Fused: rope(q) in place; rope(k) + v scattered straight into the paged
    cache (quantizing when the cache is fp8_e4m3fn). One kernel per layer
    instead of three."""
    if q.is_cuda:
        ext = _require_ext("rope_and_cache")
        ext.rope_and_cache(
            q, k, v, k_cache, v_cache, positions.to(torch.int32), cos_sin,
            slot_mapping.to(torch.int64), is_neox, k_scale, v_scale,
        )
        return
    ref.rope_inplace(q, k, positions, cos_sin, is_neox)
    ref.reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)


def reshape_and_cache(
    k: torch.Tensor,
    v: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    slot_mapping: torch.Tensor,
) -> None:
    if k.is_cuda:
        ext = _require_ext("reshape_and_cache")
        ext.reshape_and_cache(
            k.contiguous(), v.contiguous(), k_cache, v_cache, slot_mapping.to(torch.int64)
        )
        return
    ref.reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)


def mla_reshape_and_cache(
    kv_latent: torch.Tensor,
    k_rope: torch.Tensor,
    cache: torch.Tensor,
    slot_mapping: torch.Tensor,
) -> None:
    if kv_latent.is_cuda:
        ext = _require_ext("mla_reshape_and_cache")
        ext.mla_reshape_and_cache(
            kv_latent.contiguous(), k_rope.contiguous(), cache, slot_mapping.to(torch.int64)
        )
        return
    ref.mla_reshape_and_cache(kv_latent, k_rope, cache, slot_mapping)


def mla_rope_and_cache(
    q_pe: torch.Tensor,        # [T, H, DR] (a view into q)
    kv: torch.Tensor,          # [T, R + DR]
    norm_weight: torch.Tensor,  # [R]
    eps: float,
    positions: torch.Tensor,
    cos_sin: torch.Tensor,
    cache: torch.Tensor,
    slot_mapping: torch.Tensor,
    is_neox: bool = True,
) -> Optional[torch.Tensor]:
    """q_pe rotated, as rows of its own; kv's latent, RMS-normed, and its rotated key
    into the latent cache, in one launch. None where there is no kernel (CPU, other
    types, layouts or a gradient to be taken)."""
    if not q_pe.is_cuda or (torch.is_grad_enabled() and (
            q_pe.requires_grad or kv.requires_grad or norm_weight.requires_grad)):
        return None
    return _require_ext("mla_rope_and_cache").mla_rope_and_cache(
        q_pe, kv, norm_weight, eps, positions.to(torch.int32), cos_sin, cache,
        slot_mapping.to(torch.int64), is_neox)


def linear_mla_rope_and_cache(
    x: torch.Tensor, kv_weight: torch.Tensor, q_pe: torch.Tensor,
    norm_weight: torch.Tensor, eps: float, positions: torch.Tensor,
    cos_sin: torch.Tensor, cache: torch.Tensor, slot_mapping: torch.Tensor,
    is_neox: bool = True,
) -> Optional[torch.Tensor]:
    """mla_rope_and_cache() of kv = linear(x, kv_weight) of few rows: the launch that
    rotates and stores adds up the product's parts too. None where the product has no
    parts (product_has_parts()) or there is no kernel; no part of autograd."""
    if not x.is_cuda or SKINNY_GEMM_MAX_M < x.shape[0] or (
            torch.is_grad_enabled() and any(
                t.requires_grad for t in (x, kv_weight, q_pe, norm_weight))):
        return None
    return _require_ext("linear_mla_rope_and_cache").linear_mla_rope_and_cache(
        x, kv_weight, q_pe, norm_weight, eps, positions.to(torch.int32), cos_sin, cache,
        slot_mapping.to(torch.int64), is_neox)


# -- attention ---------------------------------------------------------------------


def paged_attention_decode(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_tables: torch.Tensor,
    seq_lens: torch.Tensor,
    scale: float,
    sliding_window: int = -1,
    softcap: float = 0.0,
    sinks: Optional[torch.Tensor] = None,
    max_seq_len: Optional[int] = None,
    k_scale: float = 1.0,
    v_scale: float = 1.0,
) -> torch.Tensor:
    if q.is_cuda:
        ext = _require_ext("paged_attention_decode")
        out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        if max_seq_len is None:
            max_seq_len = int(seq_lens.max().item())
        ext.paged_attention_decode(
            out,
            q,
            k_cache,
            v_cache,
            block_tables.to(torch.int32),
            seq_lens.to(torch.int32),
            scale,
            sliding_window,
            softcap,
            sinks if sinks is not None else q.new_empty(0),
            max_seq_len,
            k_scale,
            v_scale,
        )
        return out
    return ref.paged_attention_decode(
        q, k_cache, v_cache, block_tables, seq_lens, scale, sliding_window, softcap, sinks
    )


def rope_cache_attention_decode(
    q: torch.Tensor,             # [B, Hq, D] (rows may be strided, e.g. QKV views)
    k: torch.Tensor,             # [B, Hk, D]
    v: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    positions: torch.Tensor,
    cos_sin: torch.Tensor,
    slot_mapping: torch.Tensor,
    block_tables: torch.Tensor,
    seq_lens: torch.Tensor,
    scale: float,
    sliding_window: int = -1,
    sinks: Optional[torch.Tensor] = None,
    max_seq_len: Optional[int] = None,
) -> Optional[torch.Tensor]:
    """rope_and_cache and paged_attention_decode in one, q left unrotated, for steps in
    which every row is the last token of a sequence that no other row reads, and
    slot_mapping that token's place (below 0: all of the sequence is cached). None
    where there is no kernel (CPU, other types and layouts, a gradient to be taken)."""
    if not q.is_cuda or max_seq_len is None or (torch.is_grad_enabled() and any(
            t.requires_grad for t in (q, k, v, k_cache, v_cache))):
        return None
    return _require_ext("rope_cache_attention_decode").rope_cache_attention_decode(
        q, k, v, k_cache, v_cache, positions.to(torch.int32), cos_sin,
        slot_mapping.to(torch.int64), block_tables.to(torch.int32),
        seq_lens.to(torch.int32), scale, sliding_window,
        q.new_empty(0) if sinks is None else sinks, max_seq_len)


def decode_stack_has(rows: int, hidden: int, num_heads: int, num_kv_heads: int,
                     head_dim: int, intermediate: int, max_seq_len: int) -> bool:
    """Whether decode_stack has a kernel for layers of these sizes."""
    return _require_ext("decode_stack").decode_stack_has(
        rows, hidden, num_heads, num_kv_heads, head_dim, intermediate, max_seq_len)


def decode_stack(
    x: torch.Tensor, layers: List[torch.Tensor], eps: float, num_heads: int,
    num_kv_heads: int, scale: float, positions: torch.Tensor, cos_sin: torch.Tensor,
    slot_mapping: torch.Tensor, block_tables: torch.Tensor, seq_lens: torch.Tensor,
    max_seq_len: int,
) -> Optional[Tuple[torch.Tensor, torch.Tensor]]:
    """All layers of a Llama-type stack on a decode step of a few rows, in one launch:
    (what the last layer adds, the residual stream it is added to). layers: norm weight,
    q/k/v weight, its bias (empty: none), output weight, norm weight, gate/up weight,
    down weight, K and V cache of each. Rows and slot_mapping as in
    rope_cache_attention_decode. None where there is no kernel (decode_stack.hip has the
    sizes); no part of autograd."""
    if not x.is_cuda or x.dtype != torch.bfloat16 or (torch.is_grad_enabled() and any(
            t.requires_grad for t in [x, *layers])):
        return None
    return _require_ext("decode_stack").decode_stack(
        x, layers, eps, num_heads, num_kv_heads, scale, positions, cos_sin, slot_mapping,
        block_tables, seq_lens, max_seq_len)


def prefill_attention(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_tables: torch.Tensor,
    seq_lens: torch.Tensor,
    query_lens: torch.Tensor,
    scale: float,
    sliding_window: int = -1,
    softcap: float = 0.0,
    sinks: Optional[torch.Tensor] = None,
    k_scale: float = 1.0,
    v_scale: float = 1.0,
) -> torch.Tensor:
    if q.is_cuda:
        ext = _require_ext("prefill_attention")
        out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        ext.prefill_attention(
            out,
            q,
            k_cache,
            v_cache,
            block_tables.to(torch.int32),
            seq_lens.to(torch.int32),
            query_lens.to(device=q.device, dtype=torch.int32).contiguous(),
            scale,
            sliding_window,
            softcap,
            sinks if sinks is not None else q.new_empty(0),
            k_scale,
            v_scale,
        )
        return out
    return ref.prefill_attention(
        q, k_cache, v_cache, block_tables, seq_lens, query_lens, scale,
        sliding_window, softcap, sinks,
    )


def mla_paged_attention_decode(
    q_latent: torch.Tensor,
    q_rope: torch.Tensor,
    cache: torch.Tensor,
    block_tables: torch.Tensor,
    seq_lens: torch.Tensor,
    scale: float,
    max_seq_len: Optional[int] = None,
) -> torch.Tensor:
    if q_latent.is_cuda:
        ext = _require_ext("mla_paged_attention_decode")
        out = torch.empty_like(q_latent)
        if max_seq_len is None:
            max_seq_len = int(seq_lens.max().item())
        ext.mla_paged_attention_decode(
            out, q_latent.contiguous(), q_rope.contiguous(), cache,
            block_tables.to(torch.int32), seq_lens.to(torch.int32), scale,
            max_seq_len, q_latent.new_empty(0, dtype=torch.int32),
        )
        return out
    return ref.mla_paged_attention_decode(
        q_latent, q_rope, cache, block_tables, seq_lens, scale
    )


def mla_prefill_attention(
    out: torch.Tensor,      # [T, H, dv], written
    q_nope: torch.Tensor,   # [T, H, dn]
    q_pe: torch.Tensor,     # [T, H, dr]
    rows: torch.Tensor,     # [L, r + dr] context (any type), the T rows last
    w_uk: torch.Tensor,     # [H, dn, r]
    w_uv: torch.Tensor,     # [H, dv, r]
    scale: float,
) -> bool:
    """One request's causal MLA prompt portion by the flash kernel. False: the
    caller computes it (CPU, other types or widths, or few rows on a long
    context).

    The kernel's cost is the context's expansion to per-head keys and values,
    1.2 ns a row and head; in latent space the torch operations take 0.5 ms and
    26 ps a row, head and query row. Both sides in ms at 128 heads: 1 row on
    600 0.10 / 0.47, 1 on 40,000 6.2 / 0.63, 64 on 40,000 6.4 / 9.1, 512 on
    4,000 0.75 / 7.7; at 16 heads, where 32 keys take a workgroup 1.7 us
    whatever is idle, 64 on 40,000 2.1 / 1.5 and 128 on 40,000 2.2 / 2.7."""
    if not q_nope.is_cuda:
        return False
    if not _expansion_pays(*q_nope.shape[:2], rows.shape[0]):
        return False
    ext = _require_ext("mla_prefill_attention")
    return ext.mla_prefill_attention(
        out, q_nope, q_pe.contiguous(), rows.to(q_nope.dtype).contiguous(),
        w_uk, w_uv, scale,
    )


def _expansion_pays(rows: int, heads: int, context: int) -> bool:
    return rows * min(heads, 40) >= 2048 or context * max(heads, 40) <= 1 << 18


def mla_prefill_paged(
    out: torch.Tensor,           # [T, H, dv], written
    q_nope: torch.Tensor,        # [T, H, dn]
    q_pe: torch.Tensor,          # [T, H, dr]
    cache: torch.Tensor,         # [NB, BS, r + dr]
    block_tables: torch.Tensor,  # [B, max_blocks] int32
    lens: Sequence[Tuple[int, int]],
    w_uk: torch.Tensor,          # [H, dn, r]
    w_uv: torch.Tensor,          # [H, dv, r]
    scale: float,
) -> bool:
    """mla_prefill_attention of all requests at once, lens their (portion's rows, context
    rows with them), read from the cache's pages. False: the caller goes through them one
    by one, as for a cache or a length that this does not take."""
    if not q_nope.is_cuda or not all(
            _expansion_pays(n, q_nope.shape[1], context) for n, context in lens if n):
        return False
    return _require_ext("mla_prefill_paged").mla_prefill_paged(
        out, q_nope, q_pe.contiguous(), cache, block_tables, lens, w_uk, w_uv, scale)


def dsa_paged_attention_decode(
    q_latent: torch.Tensor,
    q_rope: torch.Tensor,
    cache: torch.Tensor,
    block_tables: torch.Tensor,
    seq_lens: torch.Tensor,
    topk_indices: torch.Tensor,
    scale: float,
    max_seq_len: Optional[int] = None,
) -> torch.Tensor:
    """DeepSeek-V3.2 sparse MLA decode: attention restricted to each row's
    top-k token positions (-1 padded; a row starting -1 falls back dense)."""
    if q_latent.is_cuda:
        ext = _require_ext("dsa_paged_attention_decode")
        out = torch.empty_like(q_latent)
        if max_seq_len is None:
            max_seq_len = int(seq_lens.max().item())
        ext.mla_paged_attention_decode(
            out, q_latent.contiguous(), q_rope.contiguous(), cache,
            block_tables.to(torch.int32), seq_lens.to(torch.int32), scale,
            max(max_seq_len, topk_indices.shape[1]),
            topk_indices.to(torch.int32).contiguous(),
        )
        return out
    return ref.dsa_paged_attention_decode(
        q_latent, q_rope, cache, block_tables, seq_lens, topk_indices, scale
    )


def msa_paged_attention_decode(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_tables: torch.Tensor,
    seq_lens: torch.Tensor,
    token_positions: torch.Tensor,
    scale: float,
) -> torch.Tensor:
    """MiniMax-style sparse attention over explicit token positions."""
    if q.is_cuda:
        ext = _require_ext("msa_paged_attention_decode")
        out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        ext.msa_paged_attention_decode(
            out, q, k_cache, v_cache, block_tables.to(torch.int32),
            seq_lens.to(torch.int32),
            token_positions.to(torch.int32).contiguous(), scale,
        )
        return out
    return ref.msa_paged_attention_decode(
        q, k_cache, v_cache, block_tables, seq_lens, token_positions, scale
    )


# indexer / block-score helpers run as torch compositions on both CPU and GPU
# (GEMV-scale work; the hot sparse gathers above are the HIP kernels)
def dsa_indexer_scores(q_index, index_cache, head_weights, block_tables,
                       seq_lens, max_ctx=None):
    """Weighted relu(q.k) scores over the paged index cache (DeepSeek-V3.2
    indexer). HIP MFMA kernel on GPU for the shared-key layout; torch
    reference elsewhere (reference Metal analogue: dsa_indexer.metal).
    Pass max_ctx (e.g. the graph ctx bucket) to stay hipGraph-capturable —
    int(seq_lens.max()) syncs the host otherwise."""
    if (
        q_index.is_cuda and index_cache.dim() == 3
        and q_index.dtype == torch.bfloat16
        and index_cache.dtype == torch.bfloat16
        and q_index.shape[1] <= 64 and q_index.shape[2] in (64, 128)
    ):
        ext = _require_ext("dsa_indexer_scores")
        if max_ctx is None:
            max_ctx = int(seq_lens.max())
        return ext.dsa_indexer_scores(
            q_index, index_cache, head_weights.float(),
            block_tables.int(), seq_lens.int(), max_ctx,
        )
    return ref.dsa_indexer_scores(
        q_index, index_cache, head_weights, block_tables, seq_lens
    )


def store_indexer_cache(index_keys, index_cache, slot_mapping):
    """Scatter indexer keys by slot (pad slots -1 land in the trash block)."""
    if index_keys.is_cuda and index_keys.dtype == torch.bfloat16 \
            and index_cache.dtype == torch.bfloat16:
        ext = _require_ext("store_indexer_cache")
        bs = index_cache.shape[1]
        trash_slot = (index_cache.shape[0] - 1) * bs
        ext.store_indexer_cache(
            index_keys.reshape(index_keys.shape[0], -1),
            index_cache, slot_mapping.long(), trash_slot,
        )
        return
    ref.store_indexer_cache(index_keys, index_cache, slot_mapping)


def msa_block_scores(q, k_cache, block_tables, seq_lens, sparse_block):
    """Mean-pooled per-sparse-block K scores vs the head-mean query
    (MiniMax-M3 indexer phase 1; reference msa_indexer.metal)."""
    if q.is_cuda and q.dtype == torch.bfloat16 \
            and k_cache.dtype == torch.bfloat16 and q.shape[2] in (64, 128):
        ext = _require_ext("msa_block_scores")
        max_sb = (int(seq_lens.max()) + sparse_block - 1) // sparse_block
        return ext.msa_block_scores(
            q, k_cache, block_tables.int(), seq_lens.int(), sparse_block,
            max(1, max_sb),
        )
    return ref.msa_block_scores(q, k_cache, block_tables, seq_lens, sparse_block)


def msa_topk_tokens(block_scores, seq_lens, sparse_block, topk_blocks,
                    init_blocks=1, local_blocks=2):
    """Top-k sparse blocks expanded to sorted token positions (-1 padded),
    always keeping the init/local blocks (phase 2)."""
    if block_scores.is_cuda:
        ext = _require_ext("msa_topk_tokens")
        keep_blocks = topk_blocks + init_blocks + local_blocks
        max_sb = block_scores.shape[1]
        max_positions = min(int(seq_lens.max()),
                            min(keep_blocks, max_sb) * sparse_block)
        return ext.msa_topk_tokens(
            block_scores.float(), seq_lens.int(), sparse_block, topk_blocks,
            init_blocks, local_blocks, max(1, max_positions),
        )
    return ref.msa_topk_tokens(
        block_scores, seq_lens, sparse_block, topk_blocks, init_blocks,
        local_blocks,
    )


# -- activations ----------------------------------------------------------------------


def silu_and_mul(x: torch.Tensor) -> torch.Tensor:
    if x.is_cuda:
        ext = _require_ext("silu_and_mul")
        half = x.shape[-1] // 2
        out = x.new_empty(*x.shape[:-1], half)
        ext.silu_and_mul(out, x.contiguous())
        return out
    return ref.silu_and_mul(x)


def gelu_and_mul(x: torch.Tensor) -> torch.Tensor:
    if x.is_cuda:
        ext = _require_ext("gelu_and_mul")
        half = x.shape[-1] // 2
        out = x.new_empty(*x.shape[:-1], half)
        ext.gelu_and_mul(out, x.contiguous())
        return out
    return ref.gelu_and_mul(x)


# -- dense linear (skinny-M fast path) ------------------------------------------

# Rows of x up to which linear() and linear_fp8() try the weight-streaming kernels; 0
# leaves every product to the library. Above 128 there are some for small weights alone,
# which are tried where the limit is not below that.
SKINNY_GEMM_MAX_M = int(os.environ.get("PARALLAX_SKINNY_GEMM_MAX_M", "128"))
PIECES_MAX_M = 384  # rows, and bytes of a weight, up to which these are
PIECES_MAX_BYTES = 26_000_000
NORM_LINEAR_MAX_M = 4  # rows of x up to which norm_linear() has kernels
LT_GEMM = os.environ.get("PARALLAX_LT_GEMM", "1") != "0"
_NONE = torch.empty(0, dtype=torch.bfloat16)  # an argument that is not there
_LT_REFUSED = set()  # (N, K) shapes hipBLASLt had no algorithm for


def _few_rows(x, weight, bias=None, x_scale=None, w_scale=None, gated=False):
    """x . weight^T (+ bias) by the kernels for few rows (with the scales: of fp8
    values; gated: silu of the first half of the columns times the second), None
    where they have none for it."""
    if x.dim() != 2:
        return None
    rows = x.shape[0]  # sizes first: a prompt's layers wait for the host
    if rows > SKINNY_GEMM_MAX_M and (
            SKINNY_GEMM_MAX_M < 128 or rows > PIECES_MAX_M
            or weight.numel() * weight.element_size() > PIECES_MAX_BYTES):
        return None
    fp8 = x_scale is not None
    if not (
        (fp8 or x.dtype == weight.dtype == torch.bfloat16)
        and rows > 0
        and weight.is_contiguous()
        and x.stride(1) == 1
        and (bias is None or bias.dtype == torch.bfloat16)
    ):
        return None
    ext = _require_ext("few_rows")
    return ext.few_rows(x, weight, _NONE if bias is None else bias,
                        x_scale if fp8 else _NONE, w_scale if fp8 else _NONE, gated)


def norm_linear(
    x: torch.Tensor, residual: Optional[torch.Tensor], norm_weight: torch.Tensor,
    eps: float, weight: torch.Tensor, bias: Optional[torch.Tensor] = None,
    gated: bool = False,
) -> Optional[Tuple[torch.Tensor, torch.Tensor]]:
    """(rmsnorm(x + residual) . weight^T + bias, x + residual) of a few rows in one
    launch, as fused_add_rmsnorm and linear give them, x and residual left as they
    are; gated: silu of the first half of the columns times the second. None where
    the kernel has nothing for it, or two launches are as fast (norm_linear.hip has
    the sizes); no part of autograd."""
    args = [x, norm_weight, weight] + [t for t in (residual, bias) if t is not None]
    if not x.is_cuda or x.dim() != 2 or weight.dim() != 2 or any(
            t.dtype != torch.bfloat16 for t in args):
        return None
    if torch.is_grad_enabled() and any(t.requires_grad for t in args):
        return None
    if x.shape[1] != weight.shape[1] or SKINNY_GEMM_MAX_M < x.shape[0]:
        return None
    ext = _require_ext("norm_linear")
    none = x.new_empty(0)
    return ext.norm_linear(
        x, none if residual is None else residual, norm_weight, eps, weight,
        none if bias is None else bias, gated)


def _library_takes(x, weight):
    return (
        LT_GEMM
        and x.is_cuda
        and x.dim() == 2
        and x.dtype == torch.bfloat16
        and weight.dtype == torch.bfloat16
        and x.is_contiguous()
        and weight.is_contiguous()
        and weight.shape[0] % 8 == 0
        and weight.shape[1] % 8 == 0
        and (weight.shape[0], weight.shape[1]) not in _LT_REFUSED
    )


def linear(
    x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None
) -> torch.Tensor:
    """F.linear: weight-streaming kernels for few rows (skinny_gemm.hip has the
    sizes, with both sides measured), tuned hipBLASLt for the rest. Neither takes
    part in autograd; operands that only torch's product takes otherwise (rows
    apart, odd widths) are left to it where a gradient is asked for."""
    if x.is_cuda and not (
        torch.is_grad_enabled()
        and (x.requires_grad or weight.requires_grad
             or (bias is not None and bias.requires_grad))
        and not _library_takes(x, weight)
    ):
        out = _few_rows(x, weight, bias)
        if out is not None:
            return out
    if _library_takes(x, weight):
        # tuned hipBLASLt: the default heuristic's decode-shape tile picks
        # are ~2.5x off the weight-streaming roofline (profiles/README.md);
        # first call per shape times the heuristic candidates (engine warmup,
        # outside graph capture) and later calls replay the winner
        ext = _require_ext("lt_linear")
        try:
            y = ext.lt_linear(x, weight)
        except RuntimeError as e:
            # hipBLASLt offers no algorithm for some odd shapes: those go to
            # torch's GEMM from now on (still a vendor product, never eager math)
            if "hipblaslt" not in str(e):
                raise
            _LT_REFUSED.add((weight.shape[0], weight.shape[1]))
            return torch.nn.functional.linear(x, weight, bias)
        return y if bias is None else y + bias
    return torch.nn.functional.linear(x, weight, bias)


# -- MoE ----------------------------------------------------------------------


def fused_moe_forward(
    x: torch.Tensor,          # [T, H] bf16
    w_gate_up: torch.Tensor,  # [E, 2I, H] bf16
    w_down: torch.Tensor,     # [E, H, I] bf16
    topk_ids: torch.Tensor,   # [T, k] long
    topk_weights: torch.Tensor,  # [T, k] float
    activation: str = "silu",
    limit: float = 0.0,
    bias_gate_up: Optional[torch.Tensor] = None,  # [E, 2I] bf16 (gpt-oss)
    weight_on_input: bool = False,
) -> torch.Tensor:
    """Grouped-GEMM MoE (device-side routing; graph-capture safe). Returns
    fp32 [T, H]. weight_on_input: the routing weight multiplies the expert's
    input (its gate/up accumulators, before bias and activation) instead of
    its output."""
    assert x.is_cuda
    ext = _require_ext("moe_forward")
    return ext.moe_forward(
        x.contiguous(), w_gate_up, w_down, topk_ids.long().contiguous(),
        topk_weights.float().contiguous(), activation == "gelu", limit,
        bias_gate_up if bias_gate_up is not None else x.new_empty(0),
        bool(weight_on_input))


def linear_fp8(x: torch.Tensor, w_q: torch.Tensor, w_scale: torch.Tensor,
               bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """W8A8 dense GEMM: x quantized per-tensor on the fly (two launches, the
    scale stays on the device), then the weight-streaming kernels for few rows
    or hipBLASLt fp8. CPU fallback dequantizes (plumbing tests)."""
    if not x.is_cuda:
        w = (w_q.float() * w_scale.float()).to(torch.float32)
        y = torch.nn.functional.linear(x.float(), w).to(x.dtype)
        return y if bias is None else y + bias
    ext = _require_ext("lt_linear_fp8")
    if x.dim() != 2:
        raise ValueError(f"linear_fp8 takes rows [M, K], not {tuple(x.shape)}")
    xq, xs = ext.quantize_fp8_tensor(
        (x if x.dtype == torch.bfloat16 else x.float()).contiguous())
    return linear_fp8_quantized(xq, xs, w_q, w_scale, bias)


def linear_fp8_quantized(xq: torch.Tensor, xs: torch.Tensor, w_q: torch.Tensor,
                         w_scale: torch.Tensor,
                         bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """linear_fp8 of rows that are fp8 values with one scale already."""
    ext = _require_ext("lt_linear_fp8")
    out = _few_rows(xq, w_q, bias, xs, w_scale)
    if out is not None:
        return out
    y = ext.lt_linear_fp8(xq, w_q, xs, w_scale)
    return y if bias is None else y + bias


def silu_and_mul_fp8(x: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """silu_and_mul of bf16 rows as fp8 values with one scale, as linear_fp8 makes them
    of its result; the largest magnitude is found on the way."""
    return _require_ext("silu_and_mul_fp8").silu_and_mul_fp8(x.contiguous())


def product_has_parts(rows: int, weight: torch.Tensor) -> bool:
    """Whether the product of that many rows with weight is one that linear_norm() takes,
    by its sizes: asked first, as a prompt's layers wait for the host."""
    return 4 < rows <= SKINNY_GEMM_MAX_M and weight.is_cuda and _require_ext(
        "product_parts").product_parts(rows, weight.shape[0],
                                       weight.shape[1] * weight.element_size()) > 1


def linear_norm(
    x: torch.Tensor, weight: torch.Tensor, w_scale: Optional[torch.Tensor],
    residual: Optional[torch.Tensor], norm_weight: torch.Tensor, eps: float,
    quantize: bool = False, x_scale: Optional[torch.Tensor] = None,
) -> Optional[Tuple[torch.Tensor, Optional[torch.Tensor], Optional[torch.Tensor]]]:
    """(rmsnorm(linear(x, weight) + residual), its scale, linear(x, weight) + residual)
    of few rows, x and residual left as they are: the launch that adds up a product's
    parts normalises them too. quantize: the first as fp8 values with the scale, for
    linear_fp8_quantized. weight is bf16, or fp8 with w_scale; x_scale: x is fp8 values
    with it. None where the product has no parts; no part of autograd."""
    if not _adds_parts(x, weight, residual, norm_weight):
        return None
    none = x.new_empty(0)
    r = _require_ext("linear_norm").linear_norm(
        x, none if x_scale is None else x_scale, weight,
        none if w_scale is None else w_scale,
        none if residual is None else residual, norm_weight, eps, quantize)
    if r is None:
        return None
    return r[0], r[1] if quantize else None, None if residual is None else r[2]


def _adds_parts(x: torch.Tensor, *others: Optional[torch.Tensor]) -> bool:
    return x.is_cuda and x.dim() == 2 and x.shape[0] <= SKINNY_GEMM_MAX_M and not (
        torch.is_grad_enabled() and any(
            t.requires_grad for t in (x, *others) if t is not None))


def linear_add(
    x: torch.Tensor, weight: torch.Tensor, w_scale: Optional[torch.Tensor],
    residual: torch.Tensor, x_scale: Optional[torch.Tensor] = None,
) -> Optional[torch.Tensor]:
    """linear(x, weight) + residual of few rows, the sum by the launch that adds up the
    product's parts. Operands and None as linear_norm()."""
    if not _adds_parts(x, weight, residual):
        return None
    none = x.new_empty(0)
    return _require_ext("linear_add").linear_add(
        x, none if x_scale is None else x_scale, weight,
        none if w_scale is None else w_scale, residual)


def linear_silu_and_mul(
    x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None
) -> torch.Tensor:
    """silu_and_mul(linear(x, weight, bias)), in the product's own epilogue for
    few rows: a launch of 3.5 us less (9728 x 896, one row). Not of fp8, where
    no gain showed: 40 rows of 36864 x 7168, a layer 330 us so and 325 to 339
    apart."""
    out = _few_rows(x, weight, bias, gated=True) if x.is_cuda else None
    return silu_and_mul(linear(x, weight, bias)) if out is None else out


def mla_absorb(q_nope: torch.Tensor, w_uk: torch.Tensor) -> torch.Tensor:
    """Queries [B, H, dn] into latent space [B, H, r] through w_uk [H, dn, r],
    fp32 sums."""
    if q_nope.is_cuda and q_nope.dtype == w_uk.dtype == torch.bfloat16:
        ext = _require_ext("mla_absorb")
        out = q_nope.new_empty(*q_nope.shape[:2], w_uk.shape[2])
        if ext.mla_absorb(out, q_nope, w_uk):
            return out
    return torch.einsum(
        "bhd,hdr->bhr", q_nope.float(), w_uk.float()).to(q_nope.dtype)


def mla_project_out(out_latent: torch.Tensor, w_uv: torch.Tensor) -> torch.Tensor:
    """Latent results [B, H, r] to heads [B, H, dv] through w_uv [H, dv, r],
    fp32 sums."""
    if out_latent.is_cuda and out_latent.dtype == w_uv.dtype == torch.bfloat16:
        ext = _require_ext("mla_project")
        out = out_latent.new_empty(*out_latent.shape[:2], w_uv.shape[1])
        if ext.mla_project(out, out_latent, w_uv):
            return out
    return torch.einsum(
        "bhr,hvr->bhv", out_latent.float(), w_uv.float()).to(out_latent.dtype)


def quantize_fp8_weight(w: torch.Tensor):
    """Per-output-channel fp8-E4M3 quantization of a weight tensor whose rows
    are output channels along dim -2 ([..., N, K] -> fp8 [..., N, K] +
    fp32 dequant scale [..., N]). OCP e4m3fn — the gfx950-native encoding."""
    amax = w.float().abs().amax(dim=-1).clamp_min(1e-8)
    scale = amax / 448.0
    q = (w.float() / scale.unsqueeze(-1)).clamp(-448.0, 448.0)
    return q.to(torch.float8_e4m3fn), scale.contiguous()


def fused_moe_forward_fp8(
    x: torch.Tensor,             # [T, H] bf16
    w_gate_up: torch.Tensor,     # [E, 2I, H] fp8 e4m3
    w_gu_scale: torch.Tensor,    # [E, 2I] fp32
    w_down: torch.Tensor,        # [E, H, I] fp8 e4m3
    w_down_scale: torch.Tensor,  # [E, H] fp32
    topk_ids: torch.Tensor,      # [T, k] long
    topk_weights: torch.Tensor,  # [T, k] float
    activation: str = "silu",
    limit: float = 0.0,
) -> torch.Tensor:
    """W8A8 grouped-GEMM MoE on the fp8 MFMA path (activations quantized
    per-token on device). Returns fp32 [T, H]."""
    assert x.is_cuda
    ext = _require_ext("moe_forward_fp8")
    return ext.moe_forward_fp8(
        x.contiguous(), w_gate_up, w_gu_scale, w_down, w_down_scale,
        topk_ids.long().contiguous(), topk_weights.float().contiguous(),
        activation == "gelu", limit)


# -- sampling (torch ops; GPU path uses torch's ROCm kernels — not a hot spot
#    relative to the model forward, custom kernel is a later optimization) -------

_SAMPLE_CALLS = 0


def sample_tokens(logits, temperatures, top_ps, top_ks, min_ps,
                  generator=None):
    """Batched sampling. GPU rows with no top-k/p/min-p filtering take the
    fused one-pass gumbel-max HIP kernel (the torch composition makes ~6
    passes over the [B, vocab] buffer); filtered rows fall back to the torch
    path. Seed = generator seed + a per-call counter so repeated calls draw
    fresh noise deterministically."""
    global _SAMPLE_CALLS
    if logits.is_cuda and has_extension():
        B, V = logits.shape
        temps = [float(t) for t in temperatures]
        greedy = [t <= 0.0 for t in temps]
        need_filter = any(
            (not g) and (0 < int(k) < V or float(p) < 1.0 or float(m) > 0.0)
            for g, k, p, m in zip(greedy, top_ks, top_ps, min_ps)
        )
        if not need_filter:
            ext = _require_ext("sample_gumbel")
            _SAMPLE_CALLS += 1
            base = generator.initial_seed() if generator is not None else 0x5eed
            inv_t = torch.tensor(
                [1.0 / max(t, 1e-6) for t in temps], dtype=torch.float32,
                device=logits.device,
            )
            gmask = torch.tensor(greedy, dtype=torch.uint8,
                                 device=logits.device)
            return ext.sample_gumbel(
                logits.float().contiguous(), inv_t, gmask,
                (base + _SAMPLE_CALLS) & 0x7FFFFFFFFFFF,
            )
    return ref.sample_tokens(logits, temperatures, top_ps, top_ks, min_ps,
                             generator)


apply_penalties = ref.apply_penalties


# -- sequence mixers (extension _mix) ------------------------------------------
from .mix import (  # noqa: E402,F401
    add_layernorm,
    biased_glu,
    branch_rmsnorm_add,
    clamped_glu,
    decay_attention,
    decay_powers,
    embed_streams,
    gated_delta_rule,
    gated_rmsnorm,
    gla_recurrence,
    group_rmsnorm_add,
    has_mix_extension,
    hyper_rmsnorm,
    latent_expanded_attention,
    latent_expanded_supported,
    latent_gather,
    latent_kv_store,
    latent_window_attention,
    linear_f32,
    mingru_scan,
    mlstm,
    pair_hash_embedding,
    parallel_rmsnorm_add,
    pool_cache_update,
    qkv_store,
    relu_squared,
    rope_rows,
    rope_table,
    rotate_heads,
    route_softmax,
    row_attention,
    sandwich_rmsnorm,
    short_conv,
    softcap_logits,
    xielu,
)
