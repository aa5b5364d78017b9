"""The random numbers of sampled requests, worked out by the kernel library's host code, against Python's."""
import array
import ctypes
import itertools
import subprocess
import sys

import pytest

from pytriton_llama_amd.ops import library
from pytriton_llama_amd.sampling.sampler import uniform_for, uniform_text


@pytest.mark.parametrize("ids", [
    [0, 1, 2 ** 70, -5], ["a", "", "é€", "x" * 119, "x" * 120, "x" * 121, "y" * 300], [("chat", 3), None, 2.5, b"z"]],
    ids=["numbers", "texts", "others"])
def test_uniform_numbers_of_the_library(ids):
    """One block of the hash, its edges and several; ids of any kind."""
    for seed, step in [(0, 0), (123456789, 4095)]:
        texts = [uniform_text(seed, i, step).encode() for i in ids]
        values = array.array("f", [7.0] * (3 * len(ids)))
        ends = array.array("i", itertools.accumulate(map(len, texts)))
        rc = library.load("sampling").ptl_uniforms(ctypes.c_void_p(values.buffer_info()[0]), b"".join(texts),
                                                   ctypes.c_void_p(ends.buffer_info()[0]), len(ids))
        assert rc == 0
        want = array.array("f", [uniform_for(seed, i, step) for i in ids])
        assert values[2::3] == want and set(values[0::3]) == set(values[1::3]) == {7.0}


@pytest.mark.parametrize("package", ["sampling", "engine", "cache", "models", "parts", "ops", "weights", "config"])
def test_packages_can_be_imported_first(package):
    """Each in an interpreter of its own: none needs another to be imported before it."""
    subprocess.run([sys.executable, "-c", f"import pytriton_llama_amd.{package}"], check=True, timeout=300)


def test_the_sampler_hands_over_the_texts_of_the_numbers(monkeypatch):
    """The texts of a batch that draws on all rows are those that ``uniform_for`` makes its numbers of, which a batch with a
    greedy row takes."""
    import torch

    from pytriton_llama_amd import ops
    from pytriton_llama_amd.engine.request import Request, SamplingParams
    from pytriton_llama_amd.sampling import Sampler
    took = []
    monkeypatch.setattr(ops, "sample_rows_fits", lambda logits: True)
    monkeypatch.setattr(ops, "sample_rows", lambda logits, params, texts: took.append((list(params), texts)))
    requests = [Request(id, [1], SamplingParams(temperature=0.5, top_p=0.25, seed=seed), output=[2] * n)
                for id, seed, n in ((3, None, 0), ("chat é", None, 4), (("a", 1), 9, 2), (0, 0, 1))]
    Sampler(seed=7).sample_device(torch.zeros(4, 8), requests, ahead=2)
    [(params, texts)] = took
    assert params == [0.5, 0.25, 0.0] * 4
    assert texts == [uniform_text(7, r.id if r.params.seed is None else r.params.seed, len(r.output) + 2) for r in requests]
