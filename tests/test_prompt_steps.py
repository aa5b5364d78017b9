"""Steps of prompts in native code (models/prompt_steps.py): what can be asked without a GPU."""
import pytest

from pytriton_llama_amd.config import build_model
from pytriton_llama_amd.ops import prompt
from tiny_configs import tiny


@pytest.mark.parametrize("head_dim", [2, 16, 32, 48, 80, 112, 128, 160, 256])
def test_a_model_names_the_libraries_its_prompt_steps_launch(head_dim):
    """For every head size that such a step takes (any even one): what the runner has built and loaded before the first
    step holds all that the native calls go to."""
    cfg = dict(tiny("B")[0], head_dim=head_dim)
    named = build_model(cfg).kernel_libraries()
    assert {"prompt"} | {lib for lib, _ in prompt.ENTRIES} <= set(named)
