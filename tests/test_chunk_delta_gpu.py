"""The gated delta rule of prompt portions: the chunked matrix-core kernel against the plain token-by-token form.

Both sides hold state and results in fp32 and add in different orders. Keys are unit vectors and write strengths lie in (0, 1), so a
token's rounding errors are not amplified by later ones: over a few hundred tokens 1e-4 of the largest value is some 1600 roundings
of 2^-24, and far below what one dropped or doubled token moves. Results are rounded to bf16 (2^-8 relative, at most, where the two
sides round to different neighbours)."""

import pytest
import torch

from src.ops import seq

pytestmark = pytest.mark.gpu
LENS = [133, 1, 164, 17, 115, 97, 16]   # 77 rows a sequence: so few sequences go in chunks from 9 on
PAST = [0, 5, 7, 0, 2, 0, 3]


def _inputs(H, G, D, V, channel, lens=LENS, past=PAST):
    T, S = sum(lens), len(lens)
    unit = lambda x: x / x.norm(dim=-1, keepdim=True)
    q, k = unit(torch.randn(T, G, D)) * D ** -0.5, unit(torch.randn(T, G, D) + 0.5)   # keys that overlap
    qkv = torch.cat([q.reshape(T, -1), k.reshape(T, -1), torch.randn(T, H * V)], 1)
    beta, g = torch.rand(T, H), torch.rand(T, H)
    g[torch.rand(T, H) < 0.1] = 0.0      # states that are dropped
    slab = torch.randn(T, H * (V + D) + 24).to(torch.bfloat16)
    z = slab[:, H * V + 8: H * (V + D) + 8] if channel else None
    extra = dict(z=z, z_bias=torch.randn(H * D) - 1, A_log=torch.randn(H)) if channel else {}
    rag = (torch.cat([torch.arange(n) + p for n, p in zip(lens, past)]), torch.tensor([0] + lens).cumsum(0).int(),
           torch.randperm(S + 1)[:S].int())
    return qkv, beta if channel else torch.cat([beta, g], 1), slab[:, : H * V], torch.rand(V) + 0.5, torch.randn(S + 1, H, D, V), extra, rag


def _run(args, dims, dev, **kw):
    qkv, bg, gate, norm, state, extra, rag = args
    slab = gate._base if gate._base is not None else gate
    slab = slab.to(dev)
    to = lambda t: t.to(dev) if t._base is None else slab.as_strided(t.shape, t.stride(), t.storage_offset())
    state = state.clone().to(dev)
    out = seq.gated_delta(to(qkv), to(bg), to(gate), to(norm), 1e-6, state, *dims, seq.Ragged(*(to(t) for t in rag)),
                          **{k: to(t) for k, t in extra.items()}, **kw)
    return out.cpu().float(), state.cpu()


@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("heads,groups,dim,vdim,sigmoid", [
    (4, 2, 128, 128, False), (3, 3, 64, 64, True), (2, 1, 64, 256, False), (2, 2, 128, 64, True), (2, 1, 128, 256, True),
    (3, 1, 64, 128, False)])
def test_prompt_portions(cuda, heads, groups, dim, vdim, sigmoid, channel):
    torch.manual_seed(heads + dim + vdim)
    args, dims = _inputs(heads, groups, dim, vdim, channel), (heads, groups, dim, vdim)
    want, st = _run(args, dims, "cpu", gate_sigmoid=sigmoid, mult=0.7)
    got, st2 = _run(args, dims, cuda, gate_sigmoid=sigmoid, mult=0.7)
    assert (st2 - st).abs().max() <= 1e-4 * st.abs().max()
    assert ((got - want).abs() <= 2 ** -7 * want.abs() + 1e-4 * want.abs().max()).all()


@pytest.mark.parametrize("what", ["k", "v", "beta", "decay"])
def test_later_tokens_do_not_reach_earlier_rows(cuda, what):
    """An infinite key or value or a NaN gate changes its own row and the later ones of its sequence, no others."""
    torch.manual_seed(1)
    H, D, V, at = 2, 64, 128, 99
    args = _inputs(H, H, D, V, False, [80, 80, 80], [0, 0, 3])
    want, _ = _run(args, (H, H, D, V), cuda)
    if what in "kv":
        args[0][at, (H * D if what == "k" else 2 * H * D) + 3] = float("inf")
    else:
        args[1][at, 0 if what == "beta" else H] = float("nan")
    got, _ = _run(args, (H, H, D, V), cuda)
    keep = torch.ones(240, dtype=torch.bool)
    keep[at:160] = False
    assert torch.equal(got[keep], want[keep])
    assert torch.equal(got[at:160, V:], want[at:160, V:])
    assert not torch.isfinite(got[at, :V]).all()


@pytest.mark.parametrize("sigmoid", [False, True])
@pytest.mark.parametrize("vdim", [64, 128, 256])
def test_norm_and_gate_are_those_of_short_portions(cuda, vdim, sigmoid):
    """Norm and gate of every bf16 value, to the bit as the token-by-token kernel gives them. Every token drops the state and writes one
    value under a unit key, so that its row's result is that value exactly on either side; values of 8 bits, whose squares' sums are
    exact in any order."""
    torch.manual_seed(vdim)
    H, D = 4, 64
    gate = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    gate = gate[torch.isfinite(gate)]
    gate = torch.cat([gate, gate[:65536 - gate.numel()]]).repeat(4)[torch.randperm(4 * 65536)].view(-1, H * vdim)
    T = gate.shape[0]
    eye = torch.eye(D)[torch.arange(T) % 8].repeat(1, H)
    v = (torch.randn(T, H, 1).to(torch.bfloat16).float() * torch.ones(vdim)).view(T, -1)
    qkv, bg = torch.cat([eye, eye, v], 1).to(cuda), torch.cat([torch.ones(T, H), torch.zeros(T, H)], 1).to(cuda)
    norm = torch.rand(vdim, device=cuda) + 0.5

    def run(rows):   # the same tokens as sequences of `rows`
        S = T // rows
        rag = seq.Ragged(torch.arange(rows).repeat(S).to(cuda), (torch.arange(S + 1) * rows).int().to(cuda), torch.arange(S).int().to(cuda))
        return seq.gated_delta(qkv, bg, gate.to(cuda), norm, 1e-6, torch.zeros(S, H, D, vdim, device=cuda), H, H, D, vdim, rag,
                               gate_sigmoid=sigmoid, mult=0.7)

    chunks, tokens = run(256), run(8)   # in chunks, token by token
    assert torch.equal(chunks, tokens), ((chunks != tokens).sum().item(), T * H * vdim)


@pytest.mark.parametrize("channel", [False, True])
def test_state_is_no_further_from_64_bits_than_token_by_token(cuda, channel):
    """Portions of 32 rows from an empty state, 12 draws: the 2-norm distance of the state from a float64 evaluation, in chunks and, the
    same rows eight at a time, token by token. (0.92 of the other's, 1 % from draw to draw.)"""
    S, L, H, D = 16, 32, 16, 128
    T = S * L
    unit = lambda x: x / x.norm(dim=-1, keepdim=True)
    err = [0.0, 0.0]
    for seed in range(12):
        gen = torch.Generator(cuda).manual_seed(seed)
        f = lambda *s: torch.randn(*s, device=cuda, generator=gen)
        q, k, v, beta = unit(f(S, L, H, D)), unit(f(S, L, H, D)), f(S, L, H, D), torch.sigmoid(f(S, L, H))
        A_log = 0.5 * f(H)
        extra, bg = {}, beta
        if channel:
            z = (0.5 * f(S, L, H * D)).to(torch.bfloat16)
            extra = dict(z_bias=0.7 * f(H * D) - 2.5, A_log=A_log)
            sp = torch.nn.functional.softplus(z.double() + extra["z_bias"].double())
            dec = torch.exp(-A_log.double().exp()[:, None] * sp.view(S, L, H, D))
        else:
            dec = torch.exp(-A_log.exp() * torch.nn.functional.softplus(0.7 * f(S, L, H) - 2.5))
            bg, dec = torch.cat([beta, dec], -1), dec.double()[..., None].expand(S, L, H, D)
        want = torch.zeros(S, H, D, D, dtype=torch.float64, device=cuda)
        for t in range(L):
            want *= dec[:, t, :, :, None]
            kt = k[:, t].double()
            u = beta[:, t, :, None].double() * (v[:, t].double() - (want * kt[..., None]).sum(2))
            want += kt[..., None] * u[:, :, None]
        qkv = torch.cat([x.reshape(S, L, -1) for x in (q, k, v)], 2)
        gate, norm = torch.zeros(T, H * D, device=cuda, dtype=torch.bfloat16), torch.ones(D, device=cuda)
        for n, rows in enumerate((L, 8)):
            state = torch.zeros(S, H, D, D, device=cuda)
            for a in range(0, L, rows):
                cut = lambda x: x[:, a:a + rows].reshape(S * rows, -1).contiguous()
                rag = seq.Ragged(torch.arange(a, a + rows, device=cuda).repeat(S), (torch.arange(S + 1, device=cuda) * rows).int(),
                                 torch.arange(S, device=cuda).int())
                if channel:
                    extra["z"] = cut(z)
                seq.gated_delta(cut(qkv), cut(bg), gate[: S * rows], norm, 1e-6, state, H, H, D, D, rag, **extra)
            err[n] += ((state.double() - want).norm() / want.norm()).item() / 12
    assert err[0] <= err[1] < 2e-7, err


@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("vdim,short,fill,long", [(128, [1, 9, 27], 20, 28), (64, [64, 1, 95], 70, 96)])
@pytest.mark.parametrize("more", [33, 0])
def test_divided_steps(cuda, vdim, short, fill, long, channel, more):
    """A step of so many sequences that it may be divided by their lengths: portions on either side of the cut, some of them long enough
    for it or none."""
    torch.manual_seed(vdim)
    H, D = 8, 64
    lens = short * 12 + [long, long + more] * 6 + [fill] * 22   # 70 sequences of 8 heads
    args, dims = _inputs(H, 4, D, vdim, channel, lens, [3 * (i % 2) for i in range(len(lens))]), (H, 4, D, vdim)
    assert (21 if vdim == 128 else 96) * len(lens) > sum(lens) >= (17 if vdim == 128 else 64) * len(lens)
    want, st = _run(args, dims, "cpu")
    got, st2 = _run(args, dims, cuda)
    assert (st2 - st).abs().max() <= 1e-4 * st.abs().max()
    assert ((got - want).abs() <= 2 ** -7 * want.abs() + 1e-4 * want.abs().max()).all()
