"""The attention mixer over the paged cache."""
from __future__ import annotations

import math
from typing import List, Optional

import torch

from .. import ops
from .base import (ParamSource, Part, PendingProduct, PendingScale, WorkList, as_tensor,
                   paged_kv_spec, place, register_part)
from .linear import LINEAR_LIBRARIES, decode_copy, linear
from .rotary import RotaryEncoding


# How the attention kernels cut the query rows of a step: 16 rows a work item for the vector-FMA
# kernel (over all sequences, or over those the split-KV decode kernel does not take), 64 or 128
# for the matrix-core kernel for prompt portions.
ALL_16 = WorkList(16)
PORTIONS_16 = WorkList(16, after_decode=True)
PORTIONS_64 = WorkList(64, after_decode=True)
PORTIONS_128 = WorkList(128, after_decode=True)
STEP_DECODES = 3, 8        # decoding requests from which portions beside them go into their launch, head sizes 64 and 128


@register_part("mixer", "paged_attention")
class PagedAttention(Part):
    """Grouped-query attention: q/k/v projections without bias, a position
    encoding on q and k, the new keys and values written into cache pages, then
    every token attends its sequence's keys in the pages up to its own
    position, and the output projection (lite_llama/models/llama.py:26-62 for a
    prompt, :64-105 for one decoded token; here both are one path because the
    kernels read only the cache). scale defaults to head_dim^-0.5 (llama.py:173).

    The three projection matrices are concatenated at load into one
    [(Hq + 2 Hkv) D, hidden] matrix, rows q | k | v (the reference fuses k and
    v, lite_llama/executor/weight_convert.py:229-246)."""

    def __init__(self, hidden_size: int, num_heads: int, num_kv_heads: int, head_dim: int,
                 position: Optional[Part] = None, scale: Optional[float] = None,
                 window: Optional[int] = None,
                 q_name: str = "q_proj.weight", k_name: str = "k_proj.weight",
                 v_name: str = "v_proj.weight", o_name: str = "o_proj.weight"):
        if num_heads % num_kv_heads:
            raise ValueError(f"{num_heads} heads are not a multiple of {num_kv_heads} kv heads")
        if (head_dim % 2 and position is not None) or head_dim > 640:
            raise ValueError(f"the attention kernels take head sizes up to 640 (even ones with a "
                             f"position encoding), got {head_dim}")
        self.hidden_size, self.num_heads = int(hidden_size), int(num_heads)
        self.num_kv_heads, self.head_dim = int(num_kv_heads), int(head_dim)
        self.position = position
        self.scale = float(scale) if scale is not None else 1.0 / math.sqrt(head_dim)
        self.window = int(window) if window else None
        self.names = (q_name, k_name, v_name, o_name)
        self.sink: Optional[torch.Tensor] = None    # float32 [heads], set by a mixer that wraps this one:
                                            # the softmax denominator of head h also holds exp(sink[h])
        self.force_decode_splits = 0        # tests set it to try other splits
        self.q_size = self.num_heads * self.head_dim
        self.kv_size = self.num_kv_heads * self.head_dim
        self.qkv: Optional[torch.Tensor] = None
        self.o: Optional[torch.Tensor] = None
        self.qkv_blocked: Optional[torch.Tensor] = None          # decode copies (make_decode_copies)
        self.o_blocked: Optional[torch.Tensor] = None
        libs = ("attention", "rope", "prompt") + LINEAR_LIBRARIES    # (prompt: steps of prompts, any head size)
        if self.head_dim % 32 == 0 and self.head_dim <= 128:
            libs += ("attention_prefill", "attention_step")     # the matrix-core kernels for prompt portions
        if position is not None:
            libs += tuple(position.kernel_libraries)
        self.kernel_libraries = tuple(dict.fromkeys(libs))

    def work_lists(self):
        return (ALL_16, PORTIONS_16, PORTIONS_64, PORTIONS_128)

    def cache_spec(self):
        return paged_kv_spec(self.num_kv_heads, self.head_dim, self.window)

    @property
    def graph_capturable(self) -> bool:
        return self.position is None or getattr(self.position, "graph_capturable", True)

    def param_sources(self) -> List[ParamSource]:
        qn, kn, vn, on = self.names
        return [ParamSource(qn, (self.q_size, self.hidden_size)),
                ParamSource(kn, (self.kv_size, self.hidden_size)),
                ParamSource(vn, (self.kv_size, self.hidden_size)),
                ParamSource(on, (self.hidden_size, self.q_size))]

    def load(self, tensors, dtype, device) -> None:
        qn, kn, vn, on = self.names
        self.qkv = place(torch.cat([tensors[qn], tensors[kn], tensors[vn]], dim=0),
                         "matrix", dtype, device)
        self.o = place(tensors[on], "matrix", dtype, device)
        if self.position is not None:
            self.position.load({}, dtype, device)

    def make_decode_copies(self) -> int:
        self.qkv_blocked, self.o_blocked = decode_copy(self.qkv), decode_copy(self.o)
        return sum(t.numel() * t.element_size() for t in (self.qkv_blocked, self.o_blocked)
                   if t is not None)

    takes_pending_scale = True
    can_defer_output = True

    @property
    def _in_tiles(self) -> bool:
        """Whether the tiles know this part's position encoding: none, or the plain rotation."""
        return self.position is None or (type(self.position) is RotaryEncoding
                                         and "rotary_inv_freq" not in vars(self.position))

    def forward(self, x, ctx, cache, defer_output: bool = False):
        T = x.shape[0]
        Hq, Hkv, D = self.num_heads, self.num_kv_heads, self.head_dim
        group = ctx.groups[cache.group]
        rotary = self.position.rotary_inv_freq() if self.position is not None else None
        fused = self.position is None or rotary is not None
        scale = None
        if isinstance(x, PendingScale) and fused and ops.qkv_rope_store_fits(x.values, self.qkv, D):
            x, scale = x.values, x.scale
        x = as_tensor(x)
        if (T >= ops.TILE_MIN_ROWS and self._in_tiles and ops.qkv_rope_store_tile_fits(x, self.qkv, D)
                and (cache.k.data_ptr() | cache.v.data_ptr()) % 16 == 0):
            # some tens to hundreds of rows: projection, rotation (the step's cosines and sines) and cache write in tiles
            q = ops.qkv_rope_store_tile(x, self.qkv, self.position.table(ctx) if self.position is not None else None,
                                        group.slots if cache.writable else None, cache.k, cache.v, Hq, Hkv, D, cache.page_size)
            return self._attended(q, ctx, cache, group, defer_output)
        if fused and ops.qkv_rope_store_fits(x, self.qkv, D, self.qkv_blocked):
            # the few rows of a decode step: projection, rotation and cache write in one kernel
            q = ops.qkv_rope_store(x, self.qkv, ctx.positions, rotary,
                                   group.slots if cache.writable else None, cache.k, cache.v,
                                   Hq, Hkv, D, cache.page_size, scale, blocked=self.qkv_blocked)
            return self._attended(q, ctx, cache, group, defer_output)
        if fused and ops.qkv_rope_store_f32_fits(x, self.qkv, D):       # ... in float32
            q = ops.qkv_rope_store_f32(x, self.qkv, ctx.positions, rotary, group.slots if cache.writable else None,
                                       cache.k, cache.v, Hq, Hkv, D, cache.page_size)
            return self._attended(q, ctx, cache, group, defer_output)
        qkv = linear(x, self.qkv, blocked=self.qkv_blocked)
        q = qkv[:, :self.q_size].view(T, Hq, D)
        k = qkv[:, self.q_size:self.q_size + self.kv_size].view(T, Hkv, D)
        v = qkv[:, self.q_size + self.kv_size:].view(T, Hkv, D)
        inv_freq = None
        if self.position is not None:
            inv_freq = self.position.rotary_inv_freq()
            if inv_freq is None:
                self.position.apply(q, k, ctx.positions)
        ops.rope_store(q, k, v, ctx.positions, inv_freq,
                       group.slots if cache.writable else None, cache.k, cache.v,
                       cache.page_size)
        return self._attended(q, ctx, cache, group, defer_output)

    def _attended(self, q, ctx, cache, group, defer_output: bool):
        """The attention of the rotated queries and the output projection."""
        T, Hq, D = q.shape
        out = torch.empty((T, Hq, D), dtype=q.dtype, device=q.device)
        self.attend(out, q, cache, ctx, group)
        if defer_output:                    # (the norm that follows picks the kernels by the rows)
            return PendingProduct(out.view(T, Hq * D), self.o, self.o_blocked)
        return linear(out.view(T, Hq * D), self.o, blocked=self.o_blocked)

    # ---- which kernel takes which sequences --------------------------------------
    def decode_splits(self, ctx, n_dec: int, matrix_cores: bool, device) -> int:
        """How many workgroups share one sequence's keys: enough to fill the compute
        units a few times over, never finer than one turn of a workgroup."""
        if self.force_decode_splits:
            return self.force_decode_splits
        D = self.head_dim
        G = self.num_heads // self.num_kv_heads
        if matrix_cores:
            turn = 128                              # keys a workgroup takes per turn
            groups = self.num_kv_heads
        else:
            lpk = 1
            while lpk * 16 < D:
                lpk <<= 1
            turn = 2 * (256 // lpk)
            groups = self.num_kv_heads * (-(-G // 4))
        span = max(ctx.ctx_lens[:n_dec])
        if self.window:
            span = min(span, self.window)
        # measured on MI355X (256 compute units): the matrix-core kernel is best with about two
        # workgroups a compute unit, and without splits once the batch brings 1.75 for each
        # (batch 56 with 8 kv heads; at batch 24 to 48 two splits are 2 to 3 % of a step faster
        # than one); from 513 keys on with three where there is about one workgroup a unit, up to head size 96 (us with
        # two and three, 32 rows at 8 kv heads, contexts of 130 to 2,900 / 1,000 / 2,000 / 300 keys each; all rows, then 24
        # beside 8 empty ones, which leave at once and leave their units idle, as in the recorded step that stands for 17
        # to 32 requests: head size 64 30.0 29.3 / 19.0 18.4 / 30.4 29.5 / 11.7 11.8 and 26.8 24.5 / 17.9 17.6 / 29.1 28.0 /
        # 11.3 11.7; 96 38.5 36.9 / 25.6 25.0 / 42.8 41.6 / 14.1 14.3 and 35.7 31.8 / 25.1 24.5 / 40.4 38.1 / 13.8 14.1; but
        # 128 48.6 55.0 / 31.2 33.6 / 53.1 54.3 / 16.1 18.3 and 45.5 42.1 / 28.0 29.9 / 50.7 52.3 / 15.6 17.8. 64 rows at 4 kv
        # heads, 16 at 16 and 36 at 8 the same way); the other one with about four
        base = max(1, n_dec * groups)
        cus = ops.compute_units(device)
        if matrix_cores:
            least = 3 if D <= 96 and span > 512 and 8 * base <= 9 * cus else 2
            want = 1 if 4 * base >= 7 * cus else max(-(-2 * cus // base), least)
        else:
            want = -(-4 * cus // base)
        return max(1, min(want, -(-span // turn), 64))

    def _one_launch(self, n_dec: int, q, ctx, page_size: int) -> bool:
        """Whether decoding requests and the portions beside them are one launch (csrc/attention_step.hip has the figures): some of
        the former at least, and few blocks of the latter."""
        if n_dec < STEP_DECODES[self.head_dim > 64] or n_dec == ctx.num_seqs or not ops.attention_step_fits(
                q.dtype, self.num_heads, self.num_kv_heads, self.head_dim, page_size) or q.stride(0) % 8:
            return False
        blocks = ctx.work[PORTIONS_64][0].numel()
        return 0 < blocks * self.num_heads <= ops.compute_units(q.device) * (2 if self.head_dim <= 64 else 1)

    def attend(self, out, q, cache, ctx, group, k=None, v=None) -> None:
        """``k`` / ``v``: the pools of keys and of values, [pages, Hkv, page_size, D] each, when
        they are not the cache layer's "k" and "v" (a mixer that keeps one tensor a token and
        reads it as both)."""
        k = cache.k if k is None else k
        v = cache.v if v is None else v
        D, window = self.head_dim, self.window or 0
        n_dec = ctx.num_decode_seqs if D % 16 == 0 and D <= 256 else 0      # (else: the vector kernel)
        if n_dec and self._one_launch(n_dec, q, ctx, cache.page_size):
            ops.attention_step(out, q, k, v, ctx.q_start, ctx.ctx_len, group.block_table, n_dec, *ctx.work[PORTIONS_64],
                               self.scale, window, self.decode_splits(ctx, n_dec, True, q.device), sink=self.sink,
                               tickets=getattr(ctx, "tickets", None))
            return
        if n_dec:
            mfma = (ops.attention_decode_mfma_fits(q.dtype, self.num_heads, self.num_kv_heads, D,
                                                   cache.page_size)
                    and q.stride(0) % 8 == 0)
            ops.attention_decode(out, q, k, v, ctx.q_start, ctx.ctx_len,
                                 group.block_table, n_dec, self.scale, window,
                                 self.decode_splits(ctx, n_dec, mfma, q.device), matrix_cores=mfma,
                                 sink=self.sink, tickets=getattr(ctx, "tickets", None))
        if n_dec == ctx.num_seqs:
            return
        if (ops.attention_prefill_mfma_fits(q.dtype, self.num_kv_heads, D, cache.page_size)
                and q.stride(0) % 8 == 0):
            keys = max(ctx.ctx_lens[n_dec:])
            rows, groups = ops.attention_prefill_mfma_plan(
                q.device, self.num_heads, D, ctx.work[PORTIONS_64][0].numel(),
                ctx.work[PORTIONS_128][0].numel(), min(keys, window) if window else keys)
            ws, wo = ctx.work[PORTIONS_128 if rows == 128 else PORTIONS_64]
            # (a portion alone has about as many keys as rows: it is a prompt, or the largest piece of one. What comes
            # beside decoding requests is as often the rest of a prompt behind a long prefix)
            ops.attention_prefill_mfma(out, q, k, v, ctx.q_start, ctx.ctx_len,
                                       group.block_table, ws, wo, self.scale, window, rows, groups,
                                       sink=self.sink, longest=0 if n_dec else max(ctx.q_lens))
        else:
            ws, wo = ctx.work[PORTIONS_16 if n_dec else ALL_16]
            ops.attention_generic(out, q, k, v, ctx.q_start, ctx.ctx_len,
                                  group.block_table, ws, wo, self.scale, window, sink=self.sink)

