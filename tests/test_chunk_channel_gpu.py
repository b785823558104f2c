"""Linear attention with a decay per key channel: prompt portions in chunks on the matrix cores against a float64 evaluation.

Both sides hold the same bf16 inputs. The kernel's decays come from the hardware's exponential and logarithm, some 2^-22 of an exponent of
at most 1 per token; over a few hundred tokens a state's terms are off by 1e-5 of their size at most, and results by as much of their root
mean square. Over L tokens the roundings of the decays themselves and of the state, 2^-24 of a term each, add up to L 2^-24 at most. A dropped
or doubled token moves them by 1e-2 and more."""

import pytest
import torch
import torch.nn.functional as F

from src.ops import rec, seq

pytestmark = pytest.mark.gpu


def _inputs(lens, past, H, G, D, V, pad=0):
    T, S = sum(lens), len(lens)
    x = torch.randn(T, 2 * G * D + H * V + pad).bfloat16()[:, pad:]
    z, zb = torch.randn(T, H * D + pad).bfloat16()[:, pad:], torch.randn(H * D) + 1
    z[torch.rand(T, H * D) < 0.02] = -300.0   # channels that are dropped
    state, slots = torch.randn(S + 1, H, D, V) * 0.3, torch.randperm(S + 1)[:S].int()
    pos = torch.cat([torch.arange(n) + p for n, p in zip(lens, past)])
    return x, z, zb, state, slots, pos, torch.tensor([0] + lens).cumsum(0).int()


class _Recorded:
    """The kernels, with what gated_linear_attn says of the way it took."""

    def __init__(self, kern, said):
        self.kern, self.said = kern, said

    def __getattr__(self, name):
        f = getattr(self.kern, name)
        return (lambda *a: self.said.append(f(*a))) if name == "gated_linear_attn" else f


@pytest.fixture
def said(monkeypatch):
    out, kern = [], rec._kern
    monkeypatch.setattr(rec, "_kern", lambda: _Recorded(kern(), out))
    return out


def _run(cuda, args, H, G, D, V, scale=0.3, tau=16.0):
    x, z, zb, state, slots, pos, cu = args
    pad = x.stride(0) - x.shape[1]
    wide = lambda t: F.pad(t, (pad, 0)).to(cuda)[:, pad:]
    st = state.to(cuda)
    o, _ = rec.gated_linear_attn(wide(x), 0, G * D, 2 * G * D, None, st, None, H, G, D, V, scale, seq.Ragged(pos.to(cuda), cu.to(cuda), slots.to(cuda)),
                                 z=wide(z), z_bias=zb.to(cuda), tau=tau)
    return o.cpu(), st.cpu()


def _exact(args, H, G, D, V, scale=0.3, tau=16.0):
    x, z, zb, state, slots, pos, cu = args
    T = x.shape[0]
    q, k = (x[:, i * G * D:(i + 1) * G * D].double().view(T, G, D).repeat_interleave(H // G, 1) for i in (0, 1))
    v = x[:, 2 * G * D:].double().view(T, H, V)
    dec = torch.exp(F.logsigmoid(z.double() + zb.double()) / tau).view(T, H, D)
    out, st = torch.empty(T, H, V, dtype=torch.float64), state.double()
    for s in range(len(slots)):
        S = st[slots[s]] if pos[cu[s]] > 0 else torch.zeros(H, D, V, dtype=torch.float64)
        for t in range(int(cu[s]), int(cu[s + 1])):
            S = dec[t][:, :, None] * S + k[t][:, :, None] * v[t][:, None, :]
            out[t] = (S * (q[t] * scale)[:, :, None]).sum(1)
        st[slots[s]] = S
    return out.reshape(T, H * V), st


@pytest.mark.parametrize("H,G,D,V,pad", [(4, 4, 64, 128, 0), (3, 1, 64, 64, 1), (2, 2, 64, 256, 3), (2, 1, 128, 128, 0), (4, 2, 128, 64, 1)])
@pytest.mark.parametrize("lens,past", [([17], [0]), ([17, 1, 64, 33], [0, 4, 9, 0]), ([48, 15, 130], [2, 0, 0]), ([16], [0]), ([1000, 3], [0, 5])])
def test_portions(cuda, said, H, G, D, V, pad, lens, past):
    """(An average of 16 rows of 64 x 64 goes token by token.)"""
    torch.manual_seed(sum(lens) + D + V)
    args = _inputs(lens, past, H, G, D, V, pad)
    want, ws = _exact(args, H, G, D, V)
    got, st = _run(cuda, args, H, G, D, V)
    assert said == [lens != [16] or (D, V) != (64, 64)]
    tol = 1e-5 if max(lens) < 160 else 1e-5 + max(lens) * 2.0 ** -24
    assert (got.double() - want).abs().max() <= tol * want.square().mean().sqrt() + tol * want.abs().max()
    assert (st.double() - ws).abs().max() <= tol * ws.abs().max()


@pytest.mark.parametrize("what", ["k", "v", "z"])
def test_later_tokens_do_not_reach_earlier_rows(cuda, said, what):
    """An infinite key or value or a NaN decay changes its own row and the later ones of its sequence, no others."""
    torch.manual_seed(3)
    H, D, V, at = 2, 64, 128, 60
    args = _inputs([40, 40, 41], [0, 0, 7], H, H, D, V)
    want, ws = _run(cuda, args, H, H, D, V)
    if what == "z":
        args[1][at, 5] = float("nan")
    else:
        args[0][at, H * D + 5 if what == "k" else 2 * H * D + 5] = float("inf")
    got, st = _run(cuda, args, H, H, D, V)
    assert said == [True, True]
    keep = torch.ones(121, dtype=torch.bool)
    keep[at:80] = False
    assert torch.equal(got[keep], want[keep])
    assert torch.equal(got[at:80, V:], want[at:80, V:])
    assert not torch.isfinite(got[at:80, 5]).any()
    slot = int(args[4][1])
    assert torch.equal(st[[i for i in range(4) if i != slot]], ws[[i for i in range(4) if i != slot]]) and not torch.isfinite(st[slot, 0, :, 5]).all()


@pytest.mark.parametrize("what", ["k", "q", "v", "state", "both", "nan", "overflow"])
@pytest.mark.parametrize("H,G,D,V,pad", [(2, 2, 64, 128, 0), (3, 1, 64, 64, 1), (2, 1, 64, 256, 0), (2, 1, 128, 128, 3), (2, 2, 128, 64, 0)])
def test_infinities_are_what_they_are_token_by_token(cuda, said, H, G, D, V, pad, what):
    """Rows and states are infinite, of the right sign, or NaN exactly where the recurrence itself makes them so; all others are as near as ever."""
    torch.manual_seed(D + V)
    args = _inputs([40, 33, 41], [3, 0, 7], H, G, D, V, pad)
    x, z, _, state, slots, _, _ = args
    k0, v0 = G * D, 2 * G * D
    if what in ("k", "both"):
        x[50, k0 + 5] = float("inf")
    if what == "q":
        x[47, 3] = float("-inf")
        x[60, D - 1] = float("inf")
    if what in ("v", "both"):
        x[90, v0 + V // 2 + 1] = float("-inf")
    if what == "state":
        state[slots[0], 0, 7, 9], state[slots[1], H - 1, 1, 2] = float("inf"), float("nan")   # (the second sequence is new: its slot is not read)
    if what == "nan":
        x[70, k0] = float("nan")
        z[100, 1] = float("nan")
    if what == "overflow":
        state[slots[0], H - 1, :, 40] = 3e38
        z[:40], x[:40, : k0] = 5.0, 4.0
    want, ws = _exact(args, H, G, D, V)
    want, ws = (torch.where(t.abs() > 3.4028235e38, t.sign() * float("inf"), t) for t in (want, ws))
    got, st = _run(cuda, args, H, G, D, V)
    assert said == [True]
    if what == "state":
        assert torch.isnan(st[slots[1]]).sum() == 0
    assert not torch.isfinite(want).all()
    for g, w in ((got.double(), want), (st[slots.long()].double(), ws[slots.long()])):
        assert torch.equal(torch.isnan(g), torch.isnan(w)) and torch.equal(torch.isposinf(g), torch.isposinf(w)) and torch.equal(torch.isneginf(g), torch.isneginf(w))
        keep = torch.isfinite(w)
        small = keep & (w.abs() < 1e30)
        assert (g[small] - w[small]).abs().max() <= 1e-5 * w[small].abs().max() + 1e-5 * w[small].square().mean().sqrt()
