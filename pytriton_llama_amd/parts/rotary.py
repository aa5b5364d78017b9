"""Rotary position encoding: the frequencies, and their application to q and k."""
from __future__ import annotations

import math
from typing import Optional

import torch

from .. import ops
from .base import Part, register_part


def default_inv_freq(theta: float, dim: int) -> torch.Tensor:
    """inv_freq_j = theta^(-2j/dim), float32
    (lite_llama/models/RotaryEmbedding.py:51)."""
    return 1.0 / (theta ** (torch.arange(0, dim, 2, dtype=torch.int64).float() / dim))


def llama3_inv_freq(theta: float, dim: int, factor: float, low_freq_factor: float,
                    high_freq_factor: float, original_max_position_embeddings: int) -> torch.Tensor:
    """The llama3 rescale of the frequencies by wavelength band
    (lite_llama/models/RotaryEmbedding.py:77-100): long waves divided by
    ``factor``, short waves kept, a linear blend between the two bands."""
    inv_freq = default_inv_freq(theta, dim)
    low_wavelen = original_max_position_embeddings / low_freq_factor
    high_wavelen = original_max_position_embeddings / high_freq_factor
    wavelen = 2 * math.pi / inv_freq
    scaled = torch.where(wavelen > low_wavelen, inv_freq / factor, inv_freq)
    smooth = (original_max_position_embeddings / wavelen - low_freq_factor) / (
        high_freq_factor - low_freq_factor)
    blended = (1 - smooth) * scaled / factor + smooth * scaled
    medium = ~(wavelen < high_wavelen) & ~(wavelen > low_wavelen)
    return torch.where(medium, blended, scaled)


def banded_inv_freq(base: float, dims: int, factor: float, low: float, high: float, original: float):
    """f_i = base^(-2i/dims) rescaled by wavelength band, as Llama 3.1 does it: with l = 2 pi / f,
    waves shorter than original / high keep f, waves longer than original / low get f / factor,
    those between get (1 - s) f / factor + s f with s = (original / l - low) / (high - low).
    Worked out in float64, rounded once; float32 [dims / 2]. (llama3_inv_freq above is the same
    rule in the float32 arithmetic of the reference.)"""
    i = torch.arange(0, dims // 2, dtype=torch.float64)
    f = float(base) ** (-2.0 * i / dims)
    wave = 2.0 * math.pi / f
    s = (original / wave - low) / (high - low) if high != low else torch.ones_like(f)
    blend = (1.0 - s) * f / factor + s * f
    out = torch.where(wave < original / high, f, torch.where(wave > original / low, f / factor, blend))
    return out.to(torch.float32)


def ramp_inv_freq(base: float, dims: int, factor: float, original: float, fast: float, slow: float):
    """Frequencies that go over from the unscaled f_i = base^(-2i/dims) (fast entries) to f_i /
    factor (slow entries) along a linear ramp, and the factor on sine and cosine that goes with
    them (the "YaRN" scaling of Peng, Quesnelle, Fan and Shippole). The ramp runs between the
    entries that make ``fast`` and ``slow`` turns over ``original`` positions:
    e(t) = dims ln(original / (2 pi t)) / (2 ln base), lo = max(floor(e(fast)), 0), hi =
    min(ceil(e(slow)), dims - 1), ramp_i = clamp((i - lo) / max(hi - lo, 0.001), 0, 1).
    Returns (float32 [dims / 2], 0.1 ln(factor) + 1); worked out in float64, rounded once."""
    i = torch.arange(0, dims // 2, dtype=torch.float64)
    f = float(base) ** (-2.0 * i / dims)

    def entry(turns: float) -> float:
        return dims * math.log(original / (2 * math.pi * turns)) / (2 * math.log(base))
    lo = max(math.floor(entry(fast)), 0)
    hi = min(math.ceil(entry(slow)), dims - 1)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return (f / factor * ramp + f * (1.0 - ramp)).to(torch.float32), 0.1 * math.log(factor) + 1.0


@register_part("position", "rotary")
class RotaryEncoding(Part):
    """Rotate-half RoPE. ``rope_type`` "default" or "llama3" with its four numbers
    (lite_llama/models/RotaryEmbedding.py:103-106,133-136). The angle
    position * inv_freq and its sine and cosine are float32, as in
    RotaryEmbedding.py:200-220 (attention_scaling is 1.0 there, :48)."""
    kernel_libraries = ("rope",)

    def __init__(self, head_dim: int, theta: float, rope_type: str = "default",
                 factor: float = 1.0, low_freq_factor: float = 1.0, high_freq_factor: float = 1.0,
                 original_max_position_embeddings: int = 0):
        if head_dim % 2:
            raise ValueError(f"rotary pairs need an even head size, got {head_dim}")
        self.head_dim = int(head_dim)
        if rope_type == "default":
            inv = default_inv_freq(theta, head_dim)
        elif rope_type == "llama3":
            inv = llama3_inv_freq(theta, head_dim, factor, low_freq_factor, high_freq_factor,
                                  original_max_position_embeddings)
        else:
            raise ValueError(f"unknown rope_type {rope_type!r}")
        self.inv_freq_host = inv.float().contiguous()
        self.inv_freq: Optional[torch.Tensor] = None

    def load(self, tensors, dtype, device) -> None:
        self.inv_freq = self.inv_freq_host.to(device)

    def rotary_inv_freq(self) -> Optional[torch.Tensor]:
        return self.inv_freq

    def table(self, ctx) -> ops.RopeTable:
        """``ops.rope_table`` of the step's rows; in a model's pass over ``ctx`` made once for all of its encodings."""
        if getattr(ctx, "rotations", None) is None:
            return ops.rope_table(ctx.positions, self.inv_freq)
        return ctx.rotations.table(self, ctx.positions)

    def apply(self, q: torch.Tensor, k: torch.Tensor, positions: torch.Tensor) -> None:
        """Rotate q and k ([T, heads, D] views of one buffer) in place."""
        ops.rope_store(q, k, k, positions, self.inv_freq, None, None, None, 1, k_in_place=True)


class Rotations:
    """The cosines and sines of a step's rows for the rotary encodings of a model, while its forward runs: each from the
    frequencies that its part has on the GPU then, all by one launch."""

    def __init__(self, blocks):
        self._blocks = blocks
        self._made = {}

    def table(self, encoding: RotaryEncoding, positions: torch.Tensor) -> ops.RopeTable:
        if encoding not in self._made:
            own = encoding.inv_freq
            parts = {encoding: None}
            for block in self._blocks:
                part = getattr(getattr(block, "mixer", None), "position", None)
                if type(part) is RotaryEncoding and part not in self._made and part.inv_freq is not None \
                        and part.inv_freq.shape == own.shape and part.inv_freq.device == own.device:
                    parts[part] = None
            tables = ops.rope_tables(positions, [p.inv_freq for p in parts])
            for i, part in enumerate(parts):
                self._made[part] = ops.RopeTable(tables, i)
        return self._made[encoding]
