"""Steps of prompts in native code (models/prompt_steps.py): what can be asked without a GPU."""
import ctypes

import pytest

from pytriton_llama_amd import ops
from pytriton_llama_amd.config import build_model
from pytriton_llama_amd.models import prompt_steps
from pytriton_llama_amd.ops import prompt
from tiny_configs import tiny


@pytest.mark.parametrize("head_dim", [2, 16, 32, 48, 80, 112, 128, 160, 256])
def test_a_model_names_the_libraries_its_prompt_steps_launch(head_dim):
    """For every head size that such a step takes (any even one): what the runner has built and loaded before the first
    step holds all that the native calls go to."""
    cfg = dict(tiny("B")[0], head_dim=head_dim)
    named = build_model(cfg).kernel_libraries()
    assert {"prompt"} | {lib for lib, _ in prompt.ENTRIES} <= set(named)


@pytest.mark.parametrize("part", ["block", "mixer", "feed_forward", "input_norm", "post_norm"])
def test_a_part_whose_forward_was_replaced_is_asked(part):
    """Somebody who puts a function of their own in place of a part's forward sees every step go through it: such a
    block is left to the parts."""
    block = build_model(tiny("B")[0]).blocks[0]
    assert prompt_steps._plain(block)
    watched = block if part == "block" else getattr(block, part)
    inner = watched.forward
    watched.forward = lambda *args, **kwargs: inner(*args, **kwargs)
    assert not prompt_steps._plain(block)
    del watched.forward
    assert prompt_steps._plain(block)


# what the native calls hand on, by the order of prompt.ENTRIES: p pointer, i int, l long, f float
SIGNATURES = ("pppiiilliillli" + "p", "ppplpppppiiiiiii" + "p", "pppiiilip", "ppippiifp", "ppppiifip", "pppiiilifip", "ppiiiip")
KINDS = {"p": ctypes.c_void_p, "i": ctypes.c_int, "l": ctypes.c_long, "f": ctypes.c_float}


def step_of_calls(codes, monkeypatch, tile):
    """Two layers of a step with functions of the test in place of the kernels' entries; codes: what an entry returns.
    The names called, and the error."""
    monkeypatch.setattr(prompt, "_stream", lambda: ctypes.c_void_p(0))
    called, keep = [], []
    for (lib, name), kinds in zip(prompt.ENTRIES, SIGNATURES):
        kind = ctypes.CFUNCTYPE(ctypes.c_int, *(KINDS[k] for k in kinds))
        keep.append(kind(lambda *args, name=name: called.append(name) or codes.get(name, 0)))
    table = (ctypes.c_void_p * len(keep))(*(ctypes.cast(f, ctypes.c_void_p).value for f in keep))
    step = prompt.PromptStep(70, 64, 128, 4, 2, 16, 16, 0, tile, tile, tile, 0, *[1 << 20] * 9)
    layer = prompt.PromptLayer(*[1 << 20] * 9, 1e-5, 1e-5)
    error = None
    try:
        prompt.prompt_between(table, step, None, layer)
        prompt.prompt_between(table, step, layer, layer)
        prompt.prompt_between(table, step, layer, None)
    except ops.KernelError as e:
        error = str(e)
    return called, error


@pytest.mark.parametrize("tile", [0, 2])
def test_the_entry_that_fails_in_a_native_step_is_named(monkeypatch, tile):
    called, error = step_of_calls({}, monkeypatch, tile)
    front = ["ptl_blaslt_gemm_bf16", "ptl_rope_store"]
    norm = ["ptl_tile_gemm_sums", "ptl_rows_sum_add_rmsnorm"] if tile else ["ptl_blaslt_gemm_bf16", "ptl_add_rmsnorm"]
    act = ["ptl_tile_gate_up"] if tile else ["ptl_blaslt_gemm_bf16", "ptl_silu_mul"]
    assert error is None and called == front + norm + act + norm + front + norm + act
    for name in set(called):
        for code, says in ((-1, "refused"), (-2, "launch failed")):
            got, error = step_of_calls({name: code}, monkeypatch, tile)
            assert got == called[:called.index(name) + 1]
            assert name in error and says in error


def test_arguments_of_a_native_step_that_are_refused(monkeypatch):
    monkeypatch.setattr(prompt, "_stream", lambda: ctypes.c_void_p(0))
    with pytest.raises(ops.KernelError, match="prompt_between: the kernel refused"):
        prompt.prompt_between(None, prompt.PromptStep(T=8, failed=3), None, None)
    table = (ctypes.c_void_p * len(prompt.ENTRIES))()
    with pytest.raises(ops.KernelError, match="prompt_between: the kernel refused"):
        prompt.prompt_between(table, prompt.PromptStep(T=0, failed=3), None, None)
