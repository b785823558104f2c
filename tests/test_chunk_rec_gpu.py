"""The matrix recurrences of prompt portions: the chunked matrix-core kernel against the plain token-by-token form.

Both sides hold state and results in fp32. A result is a sum of up to (tokens * dim) products of which each carries a few
2^-24 roundings, and the two sides add in different orders: 2e-5 of the largest value is some 300 such roundings, a hundred
times what is seen, and 100 times below what one dropped or doubled token moves."""

import pytest
import torch

from src.ops import lin, rec, seq

pytestmark = pytest.mark.gpu
LENS = [33, 1, 64, 31, 97, 32]
PAST = [0, 5, 7, 0, 2, 0]


def _step(dev):
    T, S = sum(LENS), len(LENS)
    cu = torch.tensor([0] + LENS).cumsum(0).int()
    pos = torch.cat([torch.arange(n) + p for n, p in zip(LENS, PAST)])
    slots = torch.randperm(S + 1)[:S].int()
    return T, S, seq.Ragged(pos.to(dev), cu.to(dev), slots.to(dev))


def _close(a, b, name):
    d, top = (a.cpu() - b.cpu()).abs().max().item(), b.abs().max().item()
    assert d <= 2e-5 * top, f"{name}: {d:.3g} of {top:.3g}"


@pytest.mark.parametrize("dim,vdim,heads,groups,norm", [
    (32, 32, 4, 1, False), (32, 32, 3, 3, True), (64, 128, 3, 3, True), (128, 64, 4, 1, False), (128, 64, 3, 1, False),
    (64, 64, 2, 2, True), (128, 128, 2, 1, True), (128, 32, 8, 2, False), (32, 128, 2, 2, False)])
def test_decay_per_head(cuda, dim, vdim, heads, groups, norm):
    torch.manual_seed(dim + vdim + heads)
    T, S, rag = _step("cpu")
    n = 2 * groups * dim + heads * vdim
    x = torch.randn(T, n + 24).to(torch.bfloat16)
    ab = torch.rand(T, heads, 3) * 2 - 0.7       # negative ones too
    ab[torch.rand(T, heads) < 0.1, 0] = 0.0      # and states that are dropped
    state, nst = torch.randn(S + 1, heads, dim, vdim), torch.randn(S + 1, heads, dim) if norm else None
    gpu = [t if t is None else t.to(cuda) for t in (x, ab, state, nst)]
    args = (16, 16 + groups * dim, 24 + 2 * groups * dim)    # v behind a gap of 8 columns
    o, nq = rec.gated_linear_attn(x, *args, ab, state, nst, heads, groups, dim, vdim, 0.3, rag)
    o2, nq2 = rec.gated_linear_attn(gpu[0], *args, gpu[1], gpu[2], gpu[3], heads, groups, dim, vdim, 0.3,
                                    seq.Ragged(*(t.to(cuda) for t in (rag.positions, rag.cu_q, rag.state_slots))))
    _close(o2, o, "results")
    _close(gpu[2], state, "state")
    if norm:
        _close(nq2, nq, "normaliser read-out")
        _close(gpu[3], nst, "normaliser")


@pytest.mark.parametrize("dim,vdim,heads", [(128, 128, 2), (64, 32, 3), (32, 64, 2)])
def test_fixed_decay_with_silu(cuda, dim, vdim, heads):
    torch.manual_seed(dim + vdim)
    T, S, rag = _step("cpu")
    x = torch.randn(T, heads * (2 * dim + vdim)).to(torch.bfloat16)
    decay, state = torch.tensor([0.999, 0.5, 0.9][:heads]), torch.randn(S + 1, heads, dim, vdim)
    st = state.to(cuda)
    o2 = lin.lightning_attn(x.to(cuda), 0, heads * dim, 2 * heads * dim, decay.to(cuda), st, heads, dim, vdim,
                            seq.Ragged(*(t.to(cuda) for t in (rag.positions, rag.cu_q, rag.state_slots))))
    o = lin.lightning_attn(x, 0, heads * dim, 2 * heads * dim, decay, state, heads, dim, vdim, rag)
    # silu(x) is rounded to bf16 on both sides; where the exponentials differ in their last bit a few inputs round the other way
    # (2^-9 of one of the summed products each)
    for a, b in ((o2.cpu(), o), (st.cpu(), state)):
        assert ((a - b).norm() / b.norm()).item() < 1e-3


@pytest.mark.parametrize("what", ["k", "v", "a", "b"])
def test_later_tokens_do_not_reach_earlier_rows(cuda, what):
    """An infinite key or value or a NaN gate changes its own row and the later ones of its sequence, no others."""
    torch.manual_seed(1)
    dim, vdim, heads, T, at = 64, 64, 2, 80, 41
    x, ab = torch.randn(T, heads * (2 * dim + vdim), device=cuda).to(torch.bfloat16), torch.rand(T, heads, 2, device=cuda)
    rag = seq.Ragged(torch.arange(40, device=cuda).repeat(2), torch.tensor([0, 40, 80], device=cuda).int(),
                     torch.tensor([1, 0], device=cuda).int())

    def run(x, ab):
        return rec.gated_linear_attn(x, 0, heads * dim, 2 * heads * dim, ab, torch.zeros(2, heads, dim, vdim, device=cuda), None,
                                     heads, heads, dim, vdim, 1.0, rag)[0]

    want = run(x, ab)
    if what in "kv":
        x[at + 9, (heads * dim if what == "k" else 2 * heads * dim) + 3] = float("inf")
    else:
        ab[at + 9, 0, "ab".index(what)] = float("nan")
    got = run(x, ab)
    assert torch.equal(got[: at + 9], want[: at + 9])
    assert not torch.isfinite(got[at + 9, :vdim]).all()


def test_silu_is_that_of_short_portions(cuda):
    """SiLU of every bf16 value as query, key and value, to the bit as the token-by-token kernel rounds it: with a decay of zero and one
    channel that is not zero a row's result is one product of three rounded values, exactly."""
    H, D, V = 4, 32, 128
    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    x = x[(x.float().abs() < 1e30) & (x.float().abs() > 1e-30)]   # (products that neither overflow nor lose bits)
    x = torch.cat([x, x])[:65536].to(cuda)
    small, decay = (x.float() < 200) & (x.float() > -30) & (x.float().abs() > 1e-6), torch.zeros(H, device=cuda)

    def run(qk, v, rows):   # qk [T, H]: channel 0 of q and k
        T = v.shape[0]
        row = torch.zeros(T, 2, H, D, dtype=torch.bfloat16, device=cuda)
        row[..., 0] = qk[:, None]
        S = T // rows
        rag = seq.Ragged(torch.arange(rows, device=cuda).repeat(S), (torch.arange(S + 1, device=cuda) * rows).int(), torch.arange(S, device=cuda).int())
        return lin.lightning_attn(torch.cat([row.view(T, -1), v], 1), 0, H * D, 2 * H * D, decay, torch.zeros(S, H, D, V, device=cuda), H, D, V, rag)

    one = torch.full((65536 // V, H), 20.0, dtype=torch.bfloat16, device=cuda)   # its SiLU is 20
    v = x.view(-1, V).repeat(1, H)[torch.arange(65536 // V, device=cuda)]
    qk, unit = torch.where(small, x, 1.0).view(-1, H), torch.full((65536 // H, H * V), 20.0, dtype=torch.bfloat16, device=cuda)
    for args in ((one, v), (qk, unit)):
        chunks, tokens = run(*args, 64), run(*args, 4)   # (below 8 rows a sequence: token by token)
        assert torch.isfinite(tokens).all()
        assert torch.equal(chunks, tokens), ((chunks != tokens).sum().item(), tokens.numel())


# portions on either side of the cut of 13 rows: a quarter of the rows in long ones, a long one alone (both divided), no long ones (not)
@pytest.mark.parametrize("lens", [[1] * 20 + [12] * 12 + [13] * 10 + [50] * 8 + [1] * 22, [8] * 70 + [13, 90], [8] * 60 + [13] * 6 + [14] * 6])
@pytest.mark.parametrize("dim,vdim", [(64, 128), (128, 128)])
def test_divided_steps(cuda, dim, vdim, lens):
    """With a normaliser, so many sequences that the step may be divided by their lengths."""
    torch.manual_seed(dim)
    heads = 16
    T, S = sum(lens), len(lens)
    assert 8 * S < T <= 10 * S and heads * S > 768
    cu = torch.tensor([0] + lens).cumsum(0).int()
    pos = torch.cat([torch.arange(n) + 3 * (i % 2) for i, n in enumerate(lens)])
    rag = seq.Ragged(pos, cu, torch.randperm(S + 1)[:S].int())
    x = torch.randn(T, heads * (2 * dim + vdim)).to(torch.bfloat16)
    ab, state, nst = torch.rand(T, heads, 3), torch.randn(S + 1, heads, dim, vdim), torch.randn(S + 1, heads, dim)
    gpu = [t.to(cuda) for t in (x, ab, state, nst)]
    at = (0, heads * dim, 2 * heads * dim)
    o, nq = rec.gated_linear_attn(x, *at, ab, state, nst, heads, heads, dim, vdim, 0.3, rag)
    o2, nq2 = rec.gated_linear_attn(gpu[0], *at, *gpu[1:], heads, heads, dim, vdim, 0.3,
                                    seq.Ragged(*(t.to(cuda) for t in (rag.positions, rag.cu_q, rag.state_slots))))
    for got, want, name in ((o2, o, "results"), (gpu[2], state, "state"), (nq2, nq, "normaliser read-out"), (gpu[3], nst, "normaliser")):
        _close(got, want, name)
