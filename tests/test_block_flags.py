"""What the model asks of its last block (models/causal_lm.py), with parts that run on the CPU: a block that replaces an
inherited forward by one with the plain signature is called with that signature."""
from types import SimpleNamespace

import pytest
import torch

from pytriton_llama_amd.models.causal_lm import CausalLM, LayerCall
from pytriton_llama_amd.parts.base import Part, says
from pytriton_llama_amd.parts.block import OutputNormBlock, ParallelResidualBlock, PreNormBlock, SandwichBlock

HIDDEN, VOCAB = 4, 7
W = torch.linspace(-1, 1, HIDDEN * VOCAB).view(VOCAB, HIDDEN)


class Embed(Part):
    def forward(self, ids):
        return torch.stack([ids.float() * (j + 1) % 5 for j in range(HIDDEN)], dim=1)


class Norm(Part):
    weight, eps, dtype = torch.ones(HIDDEN), 1e-5, torch.float32
    takes_pending_product = True

    def forward(self, x, residual, scale_ok=False):
        x = x if residual is None else x + residual
        return x / (1 + x.abs().sum(-1, keepdim=True)), x


class Mixer(Part):
    def forward(self, x, ctx, cache):
        return x.cumsum(0)


class Ffn(Part):
    def forward(self, x):
        return x * x


class Head(Part):
    vocab_size = VOCAB

    def forward(self, x):
        return (x.unsqueeze(1) * W).sum(-1)


def plain(h):
    return h + h.cumsum(0) ** 2


class PreNorm(PreNormBlock):
    def forward(self, h, residual, ctx, cache):
        return plain(h), residual


class Sandwich(SandwichBlock):
    def forward(self, h, residual, ctx, cache):
        return plain(h), residual


class OutputNorm(OutputNormBlock):
    def forward(self, h, residual, ctx, cache):
        return plain(h), residual


BLOCKS = {"prenorm": lambda c=PreNorm: c(Norm(), Mixer(), Norm(), Ffn()),
          "sandwich": lambda: Sandwich(Norm(), Mixer(), Norm()),
          "output_norm": lambda: OutputNorm(Mixer(), Norm())}


def logits(block, tokens, rows):
    model = CausalLM(None, Embed(), [block], Norm(), Head(), [], [LayerCall(0, None)], [])
    ctx = SimpleNamespace(token_ids=torch.arange(tokens, dtype=torch.int32), positions=torch.arange(tokens),
                          logit_rows=torch.tensor(rows, dtype=torch.int32), num_logit_rows=len(rows),
                          logit_rows_are_identity=rows == list(range(tokens)))
    return model.forward(ctx, SimpleNamespace(view=lambda *a: None))


@pytest.mark.parametrize("tokens,rows", [(12, [11]), (12, [3, 1]), (12, list(range(12))), (3, [0, 1, 2])])
@pytest.mark.parametrize("kind", sorted(BLOCKS))
def test_a_block_with_a_plain_forward_of_its_own(kind, tokens, rows):
    """Few rows, every row (from the number on at which the last product may go to the final norm) and a small step."""
    got = logits(BLOCKS[kind](), tokens, rows)
    h = Embed().forward(torch.arange(tokens))
    assert torch.equal(got, Head().forward(Norm().forward(plain(h)[rows], None)[0]))


@pytest.mark.parametrize("rows", [[11], list(range(12))])
def test_a_forward_replaced_on_one_block(rows):
    block = BLOCKS["prenorm"](PreNormBlock)
    inner, seen = block.forward, []

    def watched(h, residual, ctx, cache):
        seen.append(h.shape[0])
        return inner(h, residual, ctx, cache)
    want = logits(block, 12, rows)
    block.forward = watched
    assert torch.equal(logits(block, 12, rows), want) and seen == [12]


def test_blocks_of_the_package_still_give_the_wanted_rows_only():
    block = BLOCKS["prenorm"](PreNormBlock)
    sizes = []
    block.feed_forward.forward = lambda x: sizes.append(x.shape[0]) or x * x
    got = logits(block, 12, [7, 2])
    assert sizes == [2]
    assert torch.equal(got, logits(block, 12, list(range(12)))[[7, 2]])


def test_flags_and_the_forward_they_speak_of():
    class Derived(PreNormBlock):                # nothing of its own: as the class it derives from
        pass

    class Both(PreNorm):
        takes_rows = True

        def forward(self, h, residual, ctx, cache, rows=None):
            return h, residual

    class Switched(Derived):
        takes_rows = False

    make = BLOCKS["prenorm"]
    assert [says(make(c), "takes_rows") for c in (PreNormBlock, Derived, PreNorm, Both, Switched)] == [
        True, True, False, True, False]
    assert [says(make(c), "can_defer_output") for c in (Derived, PreNorm, Both)] == [True, False, False]
    assert not says(ParallelResidualBlock(HIDDEN, Mixer(), Norm()), "takes_rows")
    one = make(PreNorm)
    one.takes_rows = True
    assert says(one, "takes_rows")
