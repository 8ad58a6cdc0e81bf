"""Host side of the layer calls (csrc/torch_binding.cpp), without a GPU: what they refuse and which calls they leave to the
inner module.  A call that gets past these checks ends with the refusal of a CPU tensor."""
import pytest
import torch
import torch.fx

import tab_amd
from tab_amd import nn as tab_nn
from tab_amd.nn import TABConv2d, TABLinear, TABPackedChain


def _layer(C, KN, conv_type=tab_amd.BNN):
    words = tab_amd.operand_words(conv_type, 1, C)
    return TABConv2d(torch.zeros(KN, 3, 3, words, dtype=torch.int64), torch.zeros(KN, dtype=torch.int32), conv_type, C, KN, 3, 1, 1)


def test_chain_checks_its_layers_on_every_call():
    """A layer that reads more channels, or more planes, than the one before it wrote would read past the packed activation."""
    x = torch.zeros(1, 64, 8, 8)
    chain = TABPackedChain([_layer(64, 64), _layer(64, 64)])
    with pytest.raises(RuntimeError, match="must be a CUDA tensor"):
        chain(x)
    chain.layers[1] = _layer(640, 64)
    with pytest.raises(RuntimeError, match="64 output channels feed a layer with 640 input channels"):
        chain(x)
    chain.layers[1] = _layer(64, 64)
    chain.layers[1].conv_type = tab_amd.DRF
    with pytest.raises(RuntimeError, match="conv_type must be"):
        chain(x)
    del chain.layers[0], chain.layers[0]
    with pytest.raises(IndexError):
        chain(x)


def _linear(conv_type=tab_amd.BNN):
    words = tab_amd.operand_words(conv_type, 1, 64)
    conv = TABConv2d(torch.zeros(8, 1, 1, words, dtype=torch.int64), torch.zeros(8, dtype=torch.int32), conv_type, 64, 8, 1,
                     data_format="NHWC")
    return TABLinear(conv)


def test_linear_runs_the_inner_layers_compiled_call(monkeypatch):
    """Module.compile() replaces what calling the module runs."""
    fc, x = _linear(), torch.zeros(3, 64)
    with pytest.raises(RuntimeError, match="must be a CUDA tensor"):  # the one-call path (None: the call is left to the module)
        tab_nn._C.linear_forward(fc, tab_nn._PLAIN_CONV, x)
    monkeypatch.setattr(torch, "compile", lambda call, *args, **kwargs: lambda x: torch.full((x.shape[0], 1, 1, 8), 7.0))
    fc.conv.compile()
    assert tab_nn._C.linear_forward(fc, tab_nn._PLAIN_CONV, x) is None
    assert torch.equal(fc(x), torch.full((3, 8), 7.0))


@pytest.mark.parametrize("name", ["forward", "__call__"])
def test_linear_runs_a_method_replaced_on_the_class(monkeypatch, name):
    """Tools wrap a class's forward, or every module's __call__, to see the calls pass."""
    fc = _linear()
    monkeypatch.setattr(TABConv2d if name == "forward" else torch.nn.Module, name,
                        lambda self, x: torch.full((x.shape[0], 1, 1, 8), 7.0) if isinstance(self, TABConv2d) else self.forward(x))
    assert torch.equal(fc(torch.zeros(3, 64)), torch.full((3, 8), 7.0))


def test_linear_traces_down_to_the_inner_layer():
    """Symbolic tracing with the convolution layer as a leaf: a proxy is no tensor for the one-call path."""

    class Tracer(torch.fx.Tracer):
        def is_leaf_module(self, module, name):
            return isinstance(module, TABConv2d) or super().is_leaf_module(module, name)

    graph = Tracer().trace(_linear())
    assert [n.target for n in graph.nodes if n.op == "call_module"] == ["conv"]
    assert [n.target for n in graph.nodes if n.op == "call_method"] == ["reshape", "reshape"]
