"""Backward of the gated RMSNorm on its own, against autograd in float64: rows that
fill no workgroup, more rows than the launch has lanes for (workgroups then walk them
in several strides, the last one partly filled), and an epsilon of zero."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from gdt2_tilelang_amd.attention import _GatedNormFunction

pytestmark = pytest.mark.gpu


def _grads64(o, gate, weight, eps, dout):
    o, gate, weight = (t.double().requires_grad_(True) for t in (o, gate, weight))
    out = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + eps) * weight * F.silu(gate.reshape(o.shape))
    return torch.autograd.grad(out, (o, gate, weight), dout.double().reshape(o.shape))


@pytest.mark.parametrize("eps", [1e-5, 0.0])
@pytest.mark.parametrize("S,H,DV,dtype", [
    (1, 1, 32, torch.float32), (3, 1, 96, torch.float32), (5, 3, 128, torch.bfloat16),
    (8195, 1, 512, torch.float32),       # 4 rows a workgroup, 2048 workgroups: two strides, 3 rows in the second
    (8209, 8, 128, torch.float32),       # 16 rows a workgroup: 65672 rows, a third stride of 136
    (65537, 1, 64, torch.float16)])      # 32 rows a workgroup: one row in the second stride
def test_gated_norm_backward(S, H, DV, dtype, eps):
    print(f"gated norm backward S={S} H={H} DV={DV} {dtype} eps={eps}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(S)
    r = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    o, gate, dout = r(1, S, H, DV).to(dtype), r(1, S, H * DV).to(dtype), r(1, S, H * DV).to(dtype)
    weight = 1 + 0.1 * r(DV)
    ref = _grads64(o, gate, weight, eps, dout)
    ts = [t.clone().requires_grad_(True) for t in (o, gate, weight)]
    got = torch.autograd.grad(_GatedNormFunction.apply(*ts, eps), ts, dout)
    # per element a dozen fp32 operations and the hardware exp, rcp and rsq (2^-22), a mean of
    # DV terms, then the dtype's rounding; the weight's sums run over all rows in fp32, chains
    # of a few hundred with roundings of either sign
    tol = {torch.float32: 2e-6, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    for name, a, b, t in zip(("d_o", "d_gate", "d_weight"), got, ref, (tol, tol, 4e-6)):
        assert torch.isfinite(a).all(), name
        e = ((a.double() - b.reshape(a.shape)).norm() / b.norm()).item()
        print(f"  {name} {e:.1e}", flush=True)
        assert e < t, f"{name}: {e:.2e}"
