"""Steps of prompts in native code (models/prompt_steps.py): what can be asked without a GPU."""
import pytest

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
