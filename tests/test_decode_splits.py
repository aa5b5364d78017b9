"""How many workgroups share a decoding sequence's keys (parts/attention.py), on a device of 256 compute units."""
from types import SimpleNamespace

import pytest
import torch

from pytriton_llama_amd import ops
from pytriton_llama_amd.parts import attention
from pytriton_llama_amd.parts.attention import PagedAttention
from pytriton_llama_amd.parts.normed_attention import NormedAttention


def splits(rows, kv_heads, head_dim, longest, monkeypatch, window=None):
    monkeypatch.setattr(ops, "compute_units", lambda device: 256)
    part = PagedAttention(64, 4 * kv_heads, kv_heads, head_dim, window=window)
    ctx = SimpleNamespace(ctx_lens=[longest] + [1] * (rows - 1))
    return part.decode_splits(ctx, rows, True, "cuda")


@pytest.mark.parametrize("rows,kv_heads", [(32, 8), (33, 8), (36, 8), (64, 4), (16, 16), (18, 16), (8, 32), (128, 2)])
def test_about_one_workgroup_a_unit(rows, kv_heads, monkeypatch):
    """Three splits where they are no slower than two, full or partly empty: up to head size 96 and with more than 512
    keys. At 128 a full step loses 2 to 13 %."""
    for D in (32, 64, 96):
        assert splits(rows, kv_heads, D, 4096, monkeypatch) == 3
        assert splits(rows, kv_heads, D, 513, monkeypatch) == 3
        assert splits(rows, kv_heads, D, 512, monkeypatch) == 2
        assert splits(rows, kv_heads, D, 4096, monkeypatch, window=512) == 2
    for longest in (129, 512, 513, 4096):
        assert splits(rows, kv_heads, 128, longest, monkeypatch) == 2


@pytest.mark.parametrize("rows,kv_heads,want", [(31, 8, 3), (37, 8, 2), (48, 8, 2), (55, 8, 2), (56, 8, 1), (64, 8, 1),
                                                (16, 8, 4), (1, 8, 32), (1, 1, 32)])
@pytest.mark.parametrize("head_dim", [64, 128])
def test_other_batches(rows, kv_heads, want, head_dim, monkeypatch):
    """Two workgroups a unit, none finer than a turn of 128 keys; one from 1.75 for each on."""
    assert splits(rows, kv_heads, head_dim, 4096, monkeypatch) == want


@pytest.mark.parametrize("lengths,longest", [(dict(q_lens=[30, 300]), 300), (dict(q_lens=[]), 0), (dict(), 0)])
def test_portions_of_a_context_without_lengths(lengths, longest, monkeypatch):
    """The rows of the longest portion choose between two forms of the kernel: a context need not have them."""
    monkeypatch.setattr(ops, "compute_units", lambda device: 256)
    took = {}
    monkeypatch.setattr(ops, "attention_prefill_mfma_kv", lambda *args, **kwargs: took.update(kwargs))
    part = NormedAttention(256, 4, 2, 64, 64)
    blocks = torch.zeros(6, dtype=torch.int32)
    ctx = SimpleNamespace(num_decode_seqs=0, num_seqs=2, q_start=None, ctx_len=None, work={attention.PORTIONS_64: (blocks, blocks)},
                          **lengths)
    q = torch.zeros(330, 4, 64, dtype=torch.bfloat16)
    part.attend(torch.empty_like(q), q, SimpleNamespace(k=None, v=None, page_size=16), ctx, SimpleNamespace(block_table=None))
    assert took["longest"] == longest
