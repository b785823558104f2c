"""The selective scan of 9 - 16 states per channel over several trips of 16 tokens (4 and 16 lanes per channel; one, where waves of channels fill the SIMDs)
and one row per sequence, with rows inside wider tensors, against float64.

bf16 steps use the hardware's exponential and reciprocal (a few 2^-22) and round the result once (2^-9 of it); fp32 steps are
within some 2^-20 of the sums' terms, 1e-5 of the result's root mean square."""

import pytest
import torch
import torch.nn.functional as F

from src.ops import rec, seq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lens,I,N", [([16, 1, 50, 33], 70, 16), ([32, 15, 64], 8500, 16), ([17, 48], 4096, 11), ([47], 40, 9), ([1] * 5, 1030, 16), ([1] * 3, 65, 10),
                                      ([3, 20, 1, 17] * 6, 8500, 12), ([21, 20, 33] * 16, 8500, 16), ([2] * 32, 8500, 9)])
def test_trips_and_steps(cuda, lens, I, N, dt):
    g = torch.Generator().manual_seed(I + N)
    S, T = len(lens), sum(lens)
    x, d, z = (torch.randn(T, I + 3, generator=g).to(dt)[:, 1:I + 1] for _ in range(3))
    bc, A = torch.randn(T, 2 * N + 5, generator=g).to(dt), -torch.rand(I, N, generator=g) * 4
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
            st = torch.exp(step[:, None] * A.double()) * st + (step * x[t].double())[:, None] * bc[t, 1:N + 1].double()
            want[t] = (st @ bc[t, N + 2:2 * N + 2].double() + D.double() * x[t].double()) * F.silu(z[t].double())
        ws[slots[s]] = st
    wide = lambda v: torch.cat([torch.zeros(T, 1, dtype=dt), v, torch.zeros(T, 2, dtype=dt)], 1).to(cuda)[:, 1:I + 1]
    dev = [wide(x), wide(d), bias.to(cuda), bc.to(cuda)]
    st = state.to(cuda)
    rag = seq.Ragged(pos.to(cuda), None if max(lens) == 1 else cu.to(cuda), slots.to(cuda))
    got = rec.selective_scan(*dev, 1, N + 2, A.to(cuda), D.to(cuda), wide(z), st, rag)
    rms = want.square().mean().sqrt()
    assert ((got.cpu().double() - want).abs() <= (2 ** -8 * want.abs() if dt == torch.bfloat16 else 0) + 1e-5 * (want.abs() + rms)).all()
    assert ((st.cpu().double() - ws).abs() <= 1e-5 * (ws.abs() + ws.square().mean().sqrt())).all()
