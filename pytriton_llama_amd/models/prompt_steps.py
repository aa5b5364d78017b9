"""Prompt steps that are launched kernel by kernel: what lies between two attentions by one native call.

A step with several prompts is not recorded as a graph, and at 1B to 8B shapes Python takes longer to launch its
kernels than they take to run (csrc/prompt.hip). ``run`` goes over the blocks of such a step with one native call
and the mixer's own attention a block where they are the plain decoder's (RMSNorm, attention with rotary positions over
pages, SwiGLU, bfloat16): the same kernels in the same order with the same operands as the parts launch, so the same bits.
Everything else stays with the parts, and so does the last block, which may give some rows only. Eight prompts of 277
tokens in all at the 1B shape: 2.29 -> 1.69 ms in a row of steps, what the kernels take (one from idle takes 2.24: the host
issues it in 1.4 to 1.5).
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from .. import ops
from ..ops import kernels, prompt
from ..parts.attention import PagedAttention
from ..parts.base import PendingProduct
from ..parts.block import PreNormBlock
from ..parts.feedforward import SwiGLU
from ..parts.norm import RMSNorm
from ..parts.rotary import RotaryEncoding, Rotations


# Up to 64 rows some products go to kernels that read the decode copies of the weights.
LEAST_ROWS = 65


def _plain(block) -> bool:
    """Whether the block is the plain decoder's, and what its parts do in such a step is what their classes say: a part
    whose forward somebody replaced (to watch or to change what goes through it) is asked, not passed by."""
    mixer, ffn = block.mixer, block.feed_forward
    return (type(block) is PreNormBlock and type(mixer) is PagedAttention and type(ffn) is SwiGLU
            and type(block.input_norm) is RMSNorm and type(block.post_norm) is RMSNorm
            and block.input_norm.streams == 1 and block.post_norm.streams == 1
            and type(mixer.position) is RotaryEncoding
            and not any("forward" in vars(p) for p in (block, mixer, ffn, block.input_norm, block.post_norm))
            and "rotary_inv_freq" not in vars(mixer.position))


def _matrix(w, rows: int, cols: int) -> bool:
    return (w is not None and w.dtype == torch.bfloat16 and w.is_cuda and w.shape == (rows, cols) and w.is_contiguous()
            and w.data_ptr() % 16 == 0)


def _vector(w, n: int) -> bool:
    return w.dtype == torch.float32 and w.is_cuda and w.shape == (n,) and w.is_contiguous() and w.data_ptr() % 16 == 0


def run(model, h: torch.Tensor, ctx, storage) -> Optional[Tuple[PendingProduct, torch.Tensor]]:
    """All blocks of the run order but the last: (what they leave to the last block's first norm, the residual), or
    None where the step or a block is not of this kind."""
    T = h.shape[0]
    calls = model.schedule[:-1]
    if (T < LEAST_ROWS or not calls or h.dtype != torch.bfloat16 or h.dim() != 2
            or not h.is_cuda or not h.is_contiguous() or h.data_ptr() % 16 or kernels._timed_products):
        return None
    if not getattr(model.blocks[model.schedule[-1].block], "takes_pending_product", False):
        return None
    blocks = [model.blocks[c.block] for c in calls]
    if not all(isinstance(b, PreNormBlock) and _plain(b) for b in blocks):
        return None
    first, H = blocks[0], h.shape[1]
    mixer, ffn = first.mixer, first.feed_forward
    Hq, Hkv, D, I, act = mixer.num_heads, mixer.num_kv_heads, mixer.head_dim, ffn.intermediate_size, ffn.act
    width = (Hq + 2 * Hkv) * D
    caches = []
    for call, b in zip(calls, blocks):
        m, f = b.mixer, b.feed_forward
        cache = storage.view(call.cache_layer, call.writes)
        if ((m.num_heads, m.num_kv_heads, m.head_dim, f.intermediate_size, f.act) != (Hq, Hkv, D, I, act)
                or not _matrix(m.qkv, width, H) or not _matrix(m.o, H, Hq * D) or not _matrix(f.gate_up, 2 * I, H)
                or not _matrix(f.down, H, I) or not _vector(b.input_norm.weight, H) or not _vector(b.post_norm.weight, H)
                or not _vector(m.position.inv_freq, D // 2) or getattr(cache, "kind", "") != "paged" or not cache.writable):
            return None
        caches.append(cache)
    page_size = caches[0].page_size
    shape = (Hkv, page_size, D)
    slots = ctx.groups[caches[0].group].slots
    if (D % 2 or Hq % Hkv or H % 8 or I % 8 or width % 8 or Hq * D % 8 or ctx.positions.numel() != T
            or any(c.group != caches[0].group for c in caches)
            or any(p.dtype != torch.bfloat16 or p.dim() != 4 or p.shape[1:] != shape or not p.is_contiguous()
                   for c in caches for p in (c.k, c.v))
            or any(t.dtype != torch.int32 or t.numel() != T or not t.is_contiguous() for t in (ctx.positions, slots))):
        return None

    def rows(n):
        return torch.empty((T, n), dtype=torch.bfloat16, device=h.device)
    residual = h
    y = ops.add_rmsnorm(h, None, first.input_norm.weight, first.input_norm.eps)
    mixed, a = rows(Hq * D), rows(I)
    # which kernels take the products: what the parts would choose, asked once for all layers (their shapes are equal)
    norm = first.post_norm.weight
    o_splits = ops.gemm_tile_splits(T, H, Hq * D) if ops.gemm_tile_add_rmsnorm_fits(mixed, mixer.o, residual, norm) else 0
    down_splits = ops.gemm_tile_splits(T, H, I) if ops.gemm_tile_add_rmsnorm_fits(a, ffn.down, residual, norm) else 0
    tile = ops.gate_up_tile_fits(y, ffn.gate_up)
    qkv_tile = (ops.qkv_rope_store_tile_fits(y, mixer.qkv, D) and all(t.data_ptr() % 16 == 0 for c in caches for t in (c.k, c.v)))
    rotations = getattr(ctx, "rotations", None) or Rotations(blocks)
    tables = [rotations.table(b.mixer.position, ctx.positions) for b in blocks] if qkv_tile else [None] * len(blocks)
    # q | k | v, a product (or its float32 sums) and gate | up, one after the other in one place: each has been read when
    # the next is written, so a long step takes no more memory than by the parts, which hold the activation of the block
    # before where ``mixed`` is held here
    wide = torch.empty(T * max(width, H * max(2 * o_splits, 2 * down_splits, 1), 0 if tile else 2 * I),
                       dtype=torch.bfloat16, device=h.device)
    step = prompt.PromptStep(
        T, H, I, Hq, Hkv, D, page_size, act, o_splits, down_splits, int(tile), 0, ctx.positions.data_ptr(), slots.data_ptr(),
        y.data_ptr(), residual.data_ptr(), wide.data_ptr(), mixed.data_ptr(), wide.data_ptr(), wide.data_ptr(), a.data_ptr(),
        int(qkv_tile))
    table = prompt.entries()
    q, out = wide[:T * width].view(T, Hq + 2 * Hkv, D)[:, :Hq], mixed.view(T, Hq, D)
    before = None
    for i, (b, cache, turns) in enumerate(zip(blocks, caches, tables)):
        m, f = b.mixer, b.feed_forward
        behind = blocks[i + 1].input_norm if i + 1 < len(blocks) else b.post_norm     # (of the last one: not read)
        layer = prompt.PromptLayer(
            m.qkv.data_ptr(), m.o.data_ptr(), f.gate_up.data_ptr(), f.down.data_ptr(), m.position.inv_freq.data_ptr(),
            b.post_norm.weight.data_ptr(), behind.weight.data_ptr(), cache.k.data_ptr(), cache.v.data_ptr(),
            b.post_norm.eps, behind.eps, turns.of.address(turns.index) if turns is not None else 0)
        prompt.prompt_between(table, step, before, layer)
        m.attend(out, q, cache, ctx, ctx.groups[cache.group])
        before = layer
    prompt.prompt_between(table, step, before, None)
    last = blocks[-1].feed_forward
    return PendingProduct(a, last.down, last.down_blocked), residual
