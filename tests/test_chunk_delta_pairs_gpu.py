"""The gated delta rule of prompt portions where the products of keys, and the inverse of each chunk, come from a launch of their own, and
where they are formed inside (portions of a chunk on average, and up to two chunks with one workgroup per compute unit), against the
plain token-by-token form, with the tolerances of the chunked kernel's own tests: 1e-4 of the largest value (some 1600 roundings of 2^-24;
unit keys and write strengths in (0, 1) amplify none), results rounded to bf16."""

import pytest
import torch

from src.ops import seq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("lens,H,V", [([16] * 3, 4, 128), ([17, 15], 2, 128), ([1, 1, 64, 2, 16, 18], 2, 128), ([22] * 10, 16, 128), ([31, 1, 33, 20] * 3, 16, 64),
                                      ([48, 32, 50], 3, 256), ([16, 1, 47], 2, 256)])
def test_pairs_inside_and_apart(cuda, lens, H, V, channel):
    _against_plain(cuda, lens, H, 128, V, channel)


@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("D,V", [(64, 64), (64, 128), (64, 256), (128, 64), (128, 128), (128, 256)])
@pytest.mark.parametrize("lens,H", [([9, 9], 2), ([14, 8, 9, 5], 2), ([10] * 35, 16), ([200] + [1] * 15, 3)])
def test_short_averages(cuda, lens, H, D, V, channel):
    """From 9 rows a sequence on, with more heads than compute units later, for some widths; and where the longest is known, with the same bits."""
    one = _against_plain(cuda, lens, H, D, V, channel)
    two = _against_plain(cuda, lens, H, D, V, channel, max(lens))
    assert torch.equal(one[0], two[0]) and torch.equal(one[1], two[1])


def _against_plain(cuda, lens, H, D, V, channel, longest=0):
    torch.manual_seed(sum(lens) + V)
    S, T, G = len(lens), sum(lens), 1 if H % 2 else 2
    unit = lambda x: x / x.norm(dim=-1, keepdim=True)
    q, k = unit(torch.randn(T, G, D)) * D ** -0.5, unit(torch.randn(T, G, D) + 0.5)
    qkv = torch.cat([q.reshape(T, -1), k.reshape(T, -1), torch.randn(T, H * V)], 1)
    beta, g = torch.rand(T, H), torch.rand(T, H)
    g[torch.rand(T, H) < 0.1] = 0.0
    z = torch.randn(T, H * D + 1).to(torch.bfloat16)   # rows that start at an odd place
    extra = dict(z=z[:, 1:], z_bias=torch.randn(H * D) - 1, A_log=torch.randn(H)) if channel else {}
    gate, norm, state = torch.randn(T, H * V).to(torch.bfloat16), torch.rand(V) + 0.5, torch.randn(S + 1, H, D, V)
    rag = (torch.cat([torch.arange(n) + 3 * (i % 2) for i, n in enumerate(lens)]), torch.tensor([0] + lens).cumsum(0).int(), torch.randperm(S + 1)[:S].int())

    def run(dev):
        to = lambda t: t.to(dev)
        st, ex = state.clone().to(dev), {n: to(t) for n, t in extra.items()}
        if channel and dev != "cpu":
            ex["z"] = to(z)[:, 1:]
        out = seq.gated_delta(to(qkv), to(beta if channel else torch.cat([beta, g], 1)), to(gate), to(norm), 1e-6, st, H, G, D, V, seq.Ragged(*map(to, rag), longest), **ex)
        return out.cpu().float(), st.cpu()

    want, st = run("cpu")
    got, st2 = run(cuda)
    assert (st2 - st).abs().max() <= 1e-4 * st.abs().max()
    assert ((got - want).abs() <= 2 ** -7 * want.abs() + 1e-4 * want.abs().max()).all()
    return got, st2
