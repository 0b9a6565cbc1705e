"""The decoder's modules under symbolic tracing and scripting, which have to find the
plain operations in front of the fused kernels' dispatch."""

from __future__ import annotations

import pytest
import torch

from switchyard.model import Attention, GatedMLP, ModelConfig, RMSNorm, Rotary

CFG = ModelConfig(vocab_size=128, d_model=64, n_heads=2, d_ff=128, n_layers=2, n_blocks=2, max_seq_len=32,
                  residual="standard")


def test_a_norm_and_an_mlp_can_be_traced_symbolically():
    x = torch.randn(2, 8, 64, generator=torch.Generator().manual_seed(0))
    for module in (RMSNorm(64, 1e-6), GatedMLP(CFG)):
        traced = torch.fx.symbolic_trace(module)
        assert torch.equal(traced(x), module(x))


def test_attention_can_be_traced_around_its_rotary():
    # The rotary stays a leaf: its slice of the tables needs a concrete length.
    class Leaf(torch.fx.Tracer):
        def is_leaf_module(self, m, name):
            return isinstance(m, Rotary) or super().is_leaf_module(m, name)

    class Block(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.attn, self.rotary = Attention(CFG), Rotary(32, 32, 1e4)

        def forward(self, x):
            return self.attn(x, self.rotary)

    block = Block()
    x = torch.randn(2, 8, 64, generator=torch.Generator().manual_seed(0))
    graph = Leaf().trace(block)
    assert sum(n.op == "call_module" and n.target == "rotary" for n in graph.nodes) == 2
    assert torch.equal(torch.fx.GraphModule(block, graph)(x), block(x))
    torch.fx.symbolic_trace(block.attn)  # the rotary a proxy


@pytest.mark.filterwarnings("ignore::DeprecationWarning")
def test_a_norm_can_be_scripted():
    norm = RMSNorm(64, 1e-6)
    x = torch.randn(2, 8, 64, generator=torch.Generator().manual_seed(0))
    assert torch.equal(torch.jit.script(norm)(x), norm(x))


class _Tagged(torch.Tensor):
    """A subclass with nothing of its own but the default ``__torch_function__``, which
    keeps results in the subclass."""


def test_a_subclass_is_left_to_the_plain_operations():
    from switchyard import _lib

    x = torch.zeros(2)
    assert _lib.ordinary(x, torch.nn.Parameter(x)) and not _lib.ordinary(x, x.as_subclass(_Tagged))


@pytest.mark.gpu
@pytest.mark.parametrize("tagged", ["input", "weight"])
def test_a_subclass_comes_out_of_the_sublayers(tagged):
    x = torch.randn(2, 8, 64, generator=torch.Generator().manual_seed(0)).cuda()
    norm, mlp = RMSNorm(64, 1e-6).cuda(), GatedMLP(CFG).cuda()
    if tagged == "weight":
        norm.weight = torch.nn.Parameter(norm.weight.data.as_subclass(_Tagged))
        assert type(norm(x)) is _Tagged
    else:
        assert type(norm(x.as_subclass(_Tagged))) is _Tagged and type(mlp(x.as_subclass(_Tagged))) is _Tagged
