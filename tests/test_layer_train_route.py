"""Which training passes take the hip prologue and epilogue (decided on the host, no GPU
needed): a layer whose parts are not the ones the kernels stand in for keeps the torch
ops, which use what it has."""

from __future__ import annotations

import pytest
import torch

from gdt2_tilelang_amd import GatedDeltaNet2, GatedDeltaNet2Config


def _layer(cls=GatedDeltaNet2, conv=4):
    return cls(GatedDeltaNet2Config(hidden_size=32, num_heads=2, num_kv_heads=1, head_dim_k=64, head_dim_v=32,
                                    conv_size=conv))


X = torch.randn(2, 5, 32)


@pytest.mark.parametrize("conv", [0, 1, 4])
def test_plain_layers_take_the_kernels(conv):
    assert _layer(conv=conv)._trains_fused(X)


@pytest.mark.parametrize("name", ["_project", "_decay", "_finish"])
def test_an_overridden_method_is_called(name):
    """A subclass's (or an instance's) own projection, decay or finish is not passed by."""
    own = type("Own", (GatedDeltaNet2,), {name: lambda self, *a, **k: getattr(GatedDeltaNet2, name)(self, *a, **k)})
    assert not _layer(own)._trains_fused(X)
    layer = _layer()
    setattr(layer, name, getattr(layer, name))
    assert not layer._trains_fused(X)
    assert _layer(type("Other", (GatedDeltaNet2,), {"extra": 1}))._trains_fused(X)
