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


def _replace(layer, path, value):
    *where, name = path.split(".")
    for n in where:
        layer = getattr(layer, n)
    setattr(layer, name, value)


@pytest.mark.parametrize("path,value", [
    ("A_log", lambda: torch.nn.Parameter(torch.zeros(2))),            # more or fewer values than the kernels
    ("dt_bias", lambda: torch.nn.Parameter(torch.zeros(1, 1))),       # read, which torch broadcasts or refuses
    ("dt_bias", lambda: torch.nn.Parameter(torch.zeros(1, 64, dtype=torch.float64))),
    ("o_norm.weight", lambda: torch.nn.Parameter(torch.ones(1))),
    ("o_norm.weight", lambda: torch.nn.Parameter(torch.ones(32, device="meta"))),      # another device
    ("q_conv.conv", lambda: torch.nn.Conv1d(64, 64, 3, groups=64, padding=2)),         # another width
    ("k_conv.conv", lambda: torch.nn.Conv1d(64, 64, 4, groups=64, padding=6, dilation=2)),
    ("v_conv.conv", lambda: torch.nn.Conv1d(64, 64, 4, groups=32, padding=3)),
    ("v_conv.conv", lambda: torch.nn.Conv1d(64, 64, 4, groups=64, padding=3, padding_mode="circular"))])
def test_replaced_parts_keep_the_torch_ops(path, value):
    layer = _layer()
    _replace(layer, path, value())
    assert not layer._trains_fused(X)


@pytest.mark.gpu
@pytest.mark.parametrize("conv", [0, 4])
def test_a_projection_of_another_width_is_refused(conv):
    """As by the torch ops (a view or the conv), before any kernel reads it."""
    layer = _layer(conv=conv).cuda()
    layer.q_proj = torch.nn.Linear(32, 72, bias=False).cuda()
    assert layer._trains_fused(X.cuda())
    with pytest.raises(RuntimeError):
        layer(X.cuda())


@pytest.mark.gpu
def test_a_conv_of_another_width_still_trains():
    layer = _layer().cuda()
    for c, n in ((layer.q_conv, 64), (layer.k_conv, 64), (layer.v_conv, 64)):
        c.conv = torch.nn.Conv1d(n, n, 3, groups=n, padding=2).cuda()
    layer(X.cuda())[0].sum().backward()
    assert all(p.grad is not None and torch.isfinite(p.grad).all() for p in layer.parameters())
