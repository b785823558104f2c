"""The selective scan with a channel's states on one, two and four lanes (chosen from channels and sequences) against float64.

bf16 steps use the hardware's exponential and reciprocal (a few 2^-22) and round the result once (2^-9 of it); fp32 steps are
within some 2^-20 of the sums' terms, 1e-5 of the result's root mean square."""

import pytest
import torch
import torch.nn.functional as F

from src.ops import rec, seq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("S,I,N", [(2, 300, 13), (8, 4096, 16), (9, 4096, 16), (16, 4100, 9), (17, 4096, 16), (3, 70, 8)])
def test_lanes_of_a_channel(cuda, S, I, N, dt):
    g = torch.Generator().manual_seed(S * N)
    lens = [1 + (7 * s) % 19 for s in range(S)]
    T = sum(lens)
    x, d, z = (torch.randn(T, I, generator=g).to(dt) for _ in range(3))
    bc, A = torch.randn(T, 2 * N, generator=g).to(dt), -torch.rand(I, N, generator=g) * 4
    bias, D = torch.randn(I, generator=g) - 1, torch.randn(I, generator=g)
    state = torch.randn(S + 1, I, N, generator=g)
    slots = torch.randperm(S + 1, generator=g)[:S].int()
    cu = torch.tensor([0] + lens).cumsum(0).int()
    pos = torch.cat([torch.arange(n) + (5 if s % 2 else 0) for s, n in enumerate(lens)])
    want, ws = torch.empty(T, I, dtype=torch.float64), state.double()
    for s in range(S):
        st = ws[slots[s]] if s % 2 else torch.zeros(I, N, dtype=torch.float64)
        for t in range(int(cu[s]), int(cu[s + 1])):
            step = F.softplus(d[t].double() + bias.double())
            st = torch.exp(step[:, None] * A.double()) * st + (step * x[t].double())[:, None] * bc[t, :N].double()
            want[t] = (st @ bc[t, N:].double() + D.double() * x[t].double()) * F.silu(z[t].double())
        ws[slots[s]] = st
    dev = [v.to(cuda) for v in (x, d, bias, bc, A, D, z)]
    st = state.to(cuda)
    got = rec.selective_scan(*dev[:4], 0, N, *dev[4:], st, seq.Ragged(pos.to(cuda), cu.to(cuda), slots.to(cuda)))
    rms = want.square().mean().sqrt()
    assert ((got.cpu().double() - want).abs() <= (2 ** -8 * want.abs() if dt == torch.bfloat16 else 0) + 1e-5 * (want.abs() + rms)).all()
    assert ((st.cpu().double() - ws).abs() <= 1e-5 * (ws.abs() + ws.square().mean().sqrt())).all()
