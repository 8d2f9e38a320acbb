"""The short route of the decode calls and the packed offsets' copy, on the GPU.

A decode call whose tensors can go to the kernel as they are skips the general
path's conversions; the launch is the same, so every output and state has to be
the same bits as the general path's (taken here through a transposed copy of one
input, which has to be made contiguous first), and what the general path refuses
is still refused.
"""

import pytest
import torch

from gdt2_tilelang_amd import gdn2_attention, gdn2_decode, gdn2_decode_step

pytestmark = pytest.mark.gpu


def _inputs(lead, HK, H, DK, DV, dtype, seed=0):
    gen = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen)
    q, k = (torch.nn.functional.normalize(r(*lead, HK, DK), dim=-1).to(dtype) for _ in range(2))
    v, w, b = r(*lead, H, DV).to(dtype), torch.sigmoid(r(*lead, H, DV)).to(dtype), torch.sigmoid(r(*lead, HK, DK)).to(dtype)
    return [t.cuda() for t in (q, k, v, -torch.rand(*lead, HK, DK, generator=gen), b, w)]


def _strided(t):
    """``t``'s values in a layout that is not contiguous."""
    wide = torch.empty(*t.shape[:-1], t.shape[-1] + 8, dtype=t.dtype, device=t.device)
    wide[..., :-8] = t
    return wide[..., :-8]


@pytest.mark.parametrize("B,n,HK,H,DK,DV,dtype", [
    (1, 1, 1, 1, 32, 32, torch.float32), (3, 1, 2, 6, 64, 96, torch.bfloat16), (2, 1, 4, 4, 128, 128, torch.float16),
    (1, 1, 1, 2, 256, 64, torch.bfloat16), (2, 5, 2, 4, 128, 32, torch.bfloat16),
    (2, 0, 2, 2, 64, 64, torch.float32)])
def test_decode_routes_agree(B, n, HK, H, DK, DV, dtype):
    xs = _inputs((B, n), HK, H, DK, DV, dtype)
    s0 = torch.randn(B, H, DK, DV, device="cuda")
    got = []
    for general in (False, True):
        s = s0.clone()
        o = gdn2_decode(*((_strided(xs[0]), *xs[1:]) if general else xs), s, 0.3)
        got.append((o, s))
    assert got[0][0].shape == (B, n, H, DV) and got[0][0].dtype == dtype
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    if n != 1:
        return
    s = s0.clone()
    o = gdn2_decode_step(*(t[:, 0] for t in xs), s, 0.3)
    assert o.shape == (B, H, DV) and torch.equal(o, got[0][0][:, 0]) and torch.equal(s, got[0][1])


def test_decode_refusals_stay():
    xs = _inputs((2,), 2, 2, 64, 64, torch.float32)
    s = torch.zeros(2, 2, 64, 64, device="cuda")
    bad = [([*xs[:2], xs[2][..., :48].contiguous(), *xs[3:5], xs[5][..., :48].contiguous()], s[..., :48].contiguous(),
            ValueError),                                                              # DV not a multiple of 32
           ([xs[0].half(), *xs[1:]], s, TypeError),                                   # two dtypes
           ([t.double() if i != 3 else t for i, t in enumerate(xs)], s, TypeError),   # a dtype with no kernel
           (xs, s.transpose(2, 3), ValueError),                                       # strided state
           (xs, s[:1], ValueError), (xs, s.double(), TypeError), (xs, s.cpu(), ValueError),
           ([*xs[:2], xs[2][:1], *xs[3:5], xs[5][:1]], s, ValueError),                # v of another batch
           ([t[:0] for t in xs], s[:0], RuntimeError)]                                # no rows: null pointers
    for ts, st, err in bad:
        with pytest.raises(err):
            gdn2_decode_step(*ts, st)
    torch.cuda.synchronize()
    assert not s.any()


@pytest.mark.parametrize("where,dtype", [("cpu", torch.int32), ("cpu", torch.int64), ("cuda", torch.int32)])
def test_packed_offsets_are_the_calls_own(where, dtype):
    """The offsets are checked and copied once, in the forward: a caller that reuses
    its offset tensor before the backward gets the gradients of what it called."""
    cu = torch.tensor([0, 70, 70, 133], dtype=dtype, device=where)
    xs = [t.requires_grad_() for t in _inputs((1, 133), 2, 2, 64, 64, torch.float32)]
    o, st = gdn2_attention(*xs, output_final_state=True, cu_seqlens=cu)
    cu.fill_(133)
    got = torch.autograd.grad(o.sum() + st.sum(), xs)
    want = [torch.zeros_like(t) for t in xs]
    for a, e in ((0, 70), (70, 133)):
        part = [t.detach()[:, a:e].requires_grad_() for t in xs]
        oo, ss = gdn2_attention(*part, output_final_state=True)
        assert torch.equal(o[:, a:e], oo)
        for t, d in zip(want, torch.autograd.grad(oo.sum() + ss.sum(), part)):
            t[:, a:e] = d
    for x, y in zip(got, want):   # the same kernels on the same rows, in chunks that start at the same tokens
        assert (x - y).norm() <= 1e-6 * y.norm()
