"""What lies between the attentions of a prompt step, one native call a layer (csrc/prompt.hip): its structures and
entries for ctypes."""
from __future__ import annotations

import ctypes
from typing import Optional

from . import library
from .kernels import _check, _stream

_P, _I, _F = ctypes.c_void_p, ctypes.c_int, ctypes.c_float

# the entries a layer calls, in the order of PtlPromptEntries
ENTRIES = (("blaslt", "ptl_blaslt_gemm_bf16"), ("rope", "ptl_rope_store"), ("gemm_tile", "ptl_tile_gemm_sums"),
           ("gemm_rows", "ptl_rows_sum_add_rmsnorm"), ("norm", "ptl_add_rmsnorm"), ("gemm_tile", "ptl_tile_gate_up"),
           ("activation", "ptl_silu_mul"), ("gemm_tile", "ptl_tile_qkv_rope_store"))


class PromptStep(ctypes.Structure):
    _fields_ = ([(n, _I) for n in ("T", "H", "I", "Hq", "Hkv", "D", "page_size", "act", "o_splits", "down_splits",
                                   "gate_up_tile", "failed")]
                + [(n, _P) for n in ("positions", "slots", "y", "residual", "qkv", "mixed", "product", "gate_up", "a")]
                + [("qkv_tile", _I)])


class PromptLayer(ctypes.Structure):
    _fields_ = ([(n, _P) for n in ("qkv", "o", "gate_up", "down", "inv_freq", "post_norm", "next_norm", "k_cache", "v_cache")]
                + [("post_eps", _F), ("next_eps", _F), ("turns", _P)])


def entries():
    """The addresses of the entries, for ``prompt_between``."""
    return (ctypes.c_void_p * len(ENTRIES))(*(
        ctypes.cast(getattr(library.load(lib), name), ctypes.c_void_p).value for lib, name in ENTRIES))


def prompt_between(table, step: PromptStep, before: Optional[PromptLayer], after: Optional[PromptLayer]) -> None:
    """Launch on torch's current stream what lies between the attentions of two layers; the caller has checked the
    operands and keeps them alive until it returns."""
    code = library.load("prompt").ptl_prompt_between(
        table, ctypes.byref(step), ctypes.byref(before) if before is not None else None,
        ctypes.byref(after) if after is not None else None, _stream())
    if code:
        _check(code, f"prompt_between, {ENTRIES[step.failed][1]}" if step.failed >= 0 else "prompt_between")
