"""Training backward on tensors that start anywhere in memory: views at an element's
offset are contiguous and go to the kernels as they are, which gives the same bits as
the tensors at their allocations' start."""

from __future__ import annotations

import pytest
import torch

from gdt2_tilelang_amd import _hip, chunk_gdn2_bwd, chunk_gdn2_varlen_bwd
from oracle import make_inputs

pytestmark = pytest.mark.gpu


def _at(t, off):
    """``t``'s values ``off`` elements into an allocation of their own."""
    flat = torch.full((t.numel() + 16,), float("nan"), dtype=t.dtype, device=t.device)
    v = flat[off:off + t.numel()].view(t.shape)
    v.copy_(t)
    assert v.is_contiguous() and v.data_ptr() == flat.data_ptr() + off * t.element_size()
    return v


def _inputs(B, S, H, HK, DK, DV, dtype, do_dtype, n):
    q, k, _, g, b, _ = make_inputs(B, S, HK, DK, DV, decay_scale=0.5, seed=S)
    _, _, v, _, _, w = make_inputs(B, S, H, DK, DV, seed=S + 1)
    gen = torch.Generator().manual_seed(S)
    s0, dh = (0.3 * torch.randn(n, H, DK, DV, generator=gen) for _ in range(2))
    do = torch.randn(B, S, H, DV, generator=gen)
    ins = [t.to(dtype).cuda() if i != 3 else t.cuda() for i, t in enumerate((q, k, v, g, b, w))]
    return ins, s0.cuda(), do.to(do_dtype).cuda(), dh.cuda()


@pytest.mark.parametrize("off", [1, 3, 4])
@pytest.mark.parametrize("S,H,HK,DK,DV,dtype,do_dtype", [
    (70, 2, 2, 128, 64, torch.bfloat16, torch.bfloat16), (65, 4, 2, 64, 48, torch.float16, torch.float32),
    (33, 1, 1, 32, 16, torch.float32, torch.float32), (64, 2, 1, 128, 128, torch.bfloat16, torch.float16)])
def test_offset_views(off, S, H, HK, DK, DV, dtype, do_dtype):
    print(f"offset views off={off} S={S} H={H} HK={HK} DK={DK} DV={DV} {dtype} {do_dtype}", flush=True)
    ins, s0, do, dh = _inputs(2, S, H, HK, DK, DV, dtype, do_dtype, 2)
    want = chunk_gdn2_bwd(*ins, None, s0, do, dh)
    got = chunk_gdn2_bwd(*(_at(t, off) for t in ins), None, _at(s0, off), _at(do, off), _at(dh, off))
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_offset_views_packed():
    ins, s0, do, dh = _inputs(1, 133, 2, 1, 64, 64, torch.bfloat16, torch.bfloat16, 3)
    cu = torch.tensor([0, 70, 70, 133], dtype=torch.int32)
    want = chunk_gdn2_varlen_bwd(*ins, None, cu, s0, do, dh)
    got = chunk_gdn2_varlen_bwd(*(_at(t, 1) for t in ins), None, cu, _at(s0, 1), _at(do, 1), _at(dh, 1))
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_offset_outputs_of_the_c_entry(dtype):
    B, S, H, DK, DV = 1, 70, 2, 64, 48
    ins, s0, do, dh = _inputs(B, S, H, H, DK, DV, dtype, dtype, B)
    want = chunk_gdn2_bwd(*ins, None, s0, do, dh)
    outs = [_at(torch.zeros_like(t), 3) for t in want]
    dq, dk, dv, dg, db, dw, ds0 = outs
    lib, P, code = _hip.lib(), _hip.ptr, _hip.dtype_code(dtype)
    ws = torch.empty(lib.gdn2_hip_backward_workspace_bytes(B, H, H, DK, DV, S), dtype=torch.uint8, device="cuda")
    q, k, v, g, b, w = ins
    _hip.check(lib.gdn2_hip_backward(P(q), P(k), P(v), P(g), P(b), P(w), code, DK ** -0.5, P(s0), P(do), code, P(dh),
                                     P(dq), P(dk), P(dv), P(dg), P(db), P(dw), P(ds0), P(ws), B, S, H, H, DK, DV,
                                     _hip.stream_of(q.device)), "gdn2_hip_backward")
    for a, b in zip(outs, want):
        assert torch.equal(a, b)
