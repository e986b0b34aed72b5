"""Where the layers take the one-kernel form of a linear layer and its gate."""

import pytest

from trifusion_amd.kernels.block import gated_linear_pays

# (rows, features, depth): of each neighbouring pair one side measured faster in one
# kernel, the other as the library's product and the kernel after it
FASTER = {
    "swiglu": [(1, 1408, 512), (6400, 1408, 512), (28816, 1408, 512), (64, 2816, 1024), (1616, 2816, 1024),
               (1801, 2816, 1024), (3200, 2816, 1024), (2400, 64, 1024), (160, 1024, 768)],
    "glu": [(160, 1024, 1024), (1616, 1024, 1024), (1616, 128, 512), (1616, 256, 1024), (1, 64, 128)],
}
SLOWER = {
    "swiglu": [(1, 2816, 1024), (32, 2816, 1024), (2400, 2816, 1024), (1616, 4096, 1024), (6400, 1024, 1024),
               (1616, 64, 1024), (101, 1024, 1536), (28816, 256, 1536), (1, 64, 8192), (1616, 4096, 8192)],
    "glu": [(4, 1024, 1024), (101, 1024, 1024), (12800, 512, 1024), (1024, 256, 1024), (303, 128, 512), (4, 256, 512)],
}


@pytest.mark.parametrize("kind", ["swiglu", "glu"])
def test_sizes(kind):
    assert all(gated_linear_pays(*s, kind) for s in FASTER[kind])
    assert not any(gated_linear_pays(*s, kind) for s in SLOWER[kind])


def test_a_call_that_does_more_than_the_product_is_made(monkeypatch):
    """Hooks, replaced forwards and subclasses see the layer they were put on."""
    import torch
    from torch import nn
    from torch.nn.modules import module as nn_module

    from trifusion_amd import trifusion

    monkeypatch.setattr(trifusion, "gated_linear_fits", lambda x, weight, kind: True)
    x = torch.zeros(1, 64)

    def plain():
        return nn.Linear(64, 128, bias=False)

    assert trifusion._gates(plain(), x, "glu")
    for register in ("register_forward_hook", "register_forward_pre_hook", "register_full_backward_hook"):
        layer = plain()
        getattr(layer, register)(lambda *a: None)
        assert not trifusion._gates(layer, x, "glu")
    for register in (nn_module.register_module_forward_hook, nn_module.register_module_forward_pre_hook):
        handle = register(lambda *a: None)
        try:
            assert not trifusion._gates(plain(), x, "glu")
        finally:
            handle.remove()
    layer = plain()
    layer.forward = lambda x: x
    assert not trifusion._gates(layer, x, "glu")

    class Weight(torch.Tensor):
        pass

    layer = plain()
    layer.weight = nn.Parameter(layer.weight.detach().as_subclass(Weight), requires_grad=False)
    assert type(layer.weight) is not nn.Parameter and not trifusion._gates(layer, x, "glu")
    assert not trifusion._gates(nn.Linear(64, 128), x, "glu")
    assert trifusion._gates(plain(), x, "glu")
