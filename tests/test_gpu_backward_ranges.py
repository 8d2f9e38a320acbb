"""Training backward on inputs whose rows or channels are many powers of two apart,
row by row against autograd through the float64 recurrence."""

from __future__ import annotations

import pytest
import torch

import oracle
from gdt2_tilelang_amd import chunk_gdn2_bwd

pytestmark = pytest.mark.gpu

NAMES = ("dq", "dk", "dv", "dg", "db", "dw", "dS0")


def _inputs(S, H, DK, DV, decay, seed):
    q, k, v, g, b, w = oracle.make_inputs(1, S, H, DK, DV, decay_scale=decay, seed=seed)
    gen = torch.Generator().manual_seed(seed + 1)
    s0, dh = (0.3 * torch.randn(1, H, DK, DV, generator=gen) for _ in range(2))
    return [q, k, v, g, b, w], s0, torch.randn(1, S, H, DV, generator=gen), dh


def _grads64(ins, s0, do, dh):
    ts = [t.double().requires_grad_(True) for t in (*ins, s0)]
    o, sf = oracle.recurrent_gdn2(*ts[:6], None, ts[6], True, dtype=torch.float64)
    return torch.autograd.grad((o, sf), ts, (do.double(), dh.double()))


def _grads(ins, s0, do, dh):
    got = chunk_gdn2_bwd(*(t.cuda() for t in ins), None, *(t.cuda() for t in (s0, do, dh)))
    torch.cuda.synchronize()
    return [t.double().cpu() for t in got]


def _row_errors(a, r, floor):
    """Error of each row relative to the row itself, rows below ``floor`` left out."""
    n = r.norm(dim=-1)
    return ((a - r).norm(dim=-1) / n)[n > floor]


@pytest.mark.parametrize("DK,DV", [(32, 32), (64, 48), (128, 64)])
@pytest.mark.parametrize("S,decay", [(5, 4.0), (64, 8.0), (130, 8.0), (64, 30.0)])
def test_state_gradient_by_channel(S, decay, DK, DV):
    """A channel's row of dS_0 is as small as the decay of its first tokens, down to
    2^-80 here, and as exact as a large one."""
    print(f"state gradient rows DK={DK} DV={DV} S={S} decay={decay}", flush=True)
    ins, s0, do, dh = _inputs(S, 2, DK, DV, decay, S)
    ref, got = _grads64(ins, s0, do, dh)[6], _grads(ins, s0, do, dh)[6]
    rows = ref.norm(dim=-1)
    assert rows.min() < 2.0 ** -10 * rows.max()
    # a few chained fp32 sums of up to DK + 64 products, as at one magnitude, on factors
    # e^G whose exponent (up to 150 here, a sum of fp32 decays) is exact to 2^-24 of itself
    tol = (2 * (DK + 64) + 150) * 2.0 ** -24
    e = _row_errors(got, ref, 2.0 ** -100).max().item()
    print(f"  dS0 rows {e:.2e}, {rows.max().log2():.0f} .. {rows.min().log2():.0f}", flush=True)
    assert e < tol


@pytest.mark.parametrize("DK", [32, 64, 128])
@pytest.mark.parametrize("S,nats", [(16, 5.0), (16, 1.0), (64, 5.1), (70, 4.5)])
@pytest.mark.parametrize("scale", [1.0, 1e-6, 1e-8])
def test_small_queries_and_keys_under_decay(scale, S, nats, DK):
    """dv comes from q and k alone here (no state, no state gradient), by products over
    16 rows that decay by up to 118 binary orders: relative to its size at any size of q,
    and as exact near the diagonal as without the decay."""
    print(f"small queries DK={DK} S={S} nats={nats} scale={scale}", flush=True)
    ins, s0, do, dh = _inputs(S, 2, DK, 32, 1.0, 7)
    ins[3] = -nats * (1 + 0.02 * torch.rand(ins[3].shape, generator=torch.Generator().manual_seed(1)))
    ins[0] = ins[0] * scale
    s0, dh = torch.zeros_like(s0), torch.zeros_like(dh)
    ref, got = _grads64(ins, s0, do, dh), _grads(ins, s0, do, dh)
    # sums of up to DK + 64 products in fp32, their roundings (2^-24) of either sign
    tol = (DK + 64) ** 0.5 * 2.0 ** -24
    for i in (2, 5):
        e = ((got[i] - ref[i]).norm() / ref[i].norm()).item()
        print(f"  {NAMES[i]} {e:.2e}", flush=True)
        assert e < tol


@pytest.mark.parametrize("where", ["q", "k", "v", "do"])
@pytest.mark.parametrize("S,t,DK,DV,dtype", [(128, 90, 128, 128, torch.float32), (70, 3, 64, 96, torch.bfloat16),
                                             (64, 40, 32, 48, torch.float16)])
def test_an_infinity_spoils_only_what_it_reaches(S, t, DK, DV, dtype, where):
    """One infinite input value: the gradients it is summed into are not finite, and every
    finite one is what it is without it, not a sum that has lost its other terms."""
    print(f"infinity in {where} S={S} t={t} DK={DK} DV={DV} {dtype}", flush=True)
    ins, s0, do, dh = _inputs(S, 2, DK, DV, 0.3, 11)
    ins = [x if i == 3 else x.to(dtype) for i, x in enumerate(ins)]
    do = do.to(dtype)
    want = _grads(ins, s0, do, dh)
    bad = {"q": 0, "k": 1, "v": 2}.get(where)
    x = (do if bad is None else ins[bad]).clone()
    x[0, t, 0, 5] = float("inf")
    if bad is None:
        do = x
    else:
        ins[bad] = x
    got = _grads(ins, s0, do, dh)
    tol = 2 * (DK + 64) * 2.0 ** -24 + {torch.float32: 0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    for name, a, r in zip(NAMES, got, want):
        fin = torch.isfinite(a)
        assert ((a - r).abs()[fin] <= tol * r.abs().max()).all(), name
        assert fin[..., 1, :].all() if name != "dS0" else fin[:, 1].all(), name     # the other head
    if where in ("v", "do"):                # a value column of its own in dv, dw and dS_0
        for i in (2, 5, 6):
            assert torch.isfinite(torch.cat([got[i][..., :5], got[i][..., 6:]], -1)).all(), NAMES[i]


@pytest.mark.parametrize("DK,DV", [(64, 64), (128, 128)])
@pytest.mark.parametrize("bits", [10, 24])
@pytest.mark.parametrize("state", [False, True])
def test_rows_far_apart(state, bits, DK, DV):
    """Rows of d_out and v 2^-10 and 2^-24 of the others' keep their own gradients: row by
    row as with rows of one size."""
    print(f"rows far apart DK={DK} DV={DV} bits={bits} state={state}", flush=True)
    ins, s0, do, dh = _inputs(64, 2, DK, DV, 0.3, 5)
    do[:, 32:] *= 2.0 ** -bits           # later rows: nothing of a larger one is summed into theirs
    do[:, 5:17:2] *= 2.0 ** -bits        # (dq_t = d_out_t S^T and its pairs come from row t alone)
    ins[2][:, 10:30:3] *= 2.0 ** -bits   # dw = v dY
    dh = torch.zeros_like(dh)
    s0 = s0 if state else torch.zeros_like(s0)
    ref, got = _grads64(ins, s0, do, dh), _grads(ins, s0, do, dh)
    # the largest of 100 rows' sums of up to DK + DV products, roundings of 2^-24: four
    # standard deviations
    tol = 4 * (DK + DV) ** 0.5 * 2.0 ** -24
    for i, name in enumerate(NAMES[:6]):
        a, r = (got[i], ref[i]) if name not in ("dk", "dg", "db") else (got[i][:, 32:], ref[i][:, 32:])
        e = _row_errors(a, r, 0).max().item()
        print(f"  {name} rows {e:.2e}", flush=True)
        assert e < tol, name
