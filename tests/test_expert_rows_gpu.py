"""Rows of the experts: the pairs put in order of their experts, at the edges of the kernels (2048 pairs less 8 per expert, 4096, 12288 and
32768 in one reading), and the group-limited choice, at the edges of the experts a lane holds (64, 256, 512) and with ties."""

import pytest
import torch

from src import ops
from src.ops import mix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,E", [(0, 3), (1, 1), (63, 10), (511, 8), (512, 256), (513, 64), (1920, 16), (1921, 16), (3, 256), (4097, 31), (8191, 2), (8193, 65), (20001, 256), (12289, 12), (32768, 64), (40000, 5)])
@pytest.mark.parametrize("kern", ["main", "mix"])
@pytest.mark.parametrize("lean", [1, 6])
def test_align(cuda, n, E, kern, lean):
    """Whatever the experts' shares (lean 6: most pairs to the first ones). With many pairs those of an expert ascend."""
    torch.manual_seed(n + E)
    ids = (torch.rand(n, device=cuda) ** lean * E).int().clamp_(max=E - 1)
    off, at, pos = (torch.full((s,), -7, dtype=torch.int32, device=cuda) for s in (E + 1, n, n))
    (ops if kern == "main" else mix)._kern().moe_align(off, at, pos, ids, E)
    want = torch.sort(ids.long(), stable=True).indices
    assert torch.equal(pos.long()[at.long()], torch.arange(n, device=cuda)) and torch.equal(ids[at.long()], ids[want])
    assert n + 8 * E <= 2048 or torch.equal(at.long(), want)
    assert off.tolist() == [0, *torch.bincount(ids.long(), minlength=E).cumsum(0).tolist()]


@pytest.mark.parametrize("E,k,groups,keep", [(1, 1, 1, 1), (10, 3, 5, 2), (63, 63, 1, 1), (64, 6, 4, 2), (64, 8, 64, 8), (65, 5, 13, 3), (256, 8, 8, 4),
                                             (257, 70, 1, 1), (512, 300, 4, 3), (512, 9, 512, 9)])
def test_grouped_choice(cuda, E, k, groups, keep):
    """Logits in steps of 1/4 (equal ones have equal scores, others differ by more than rounding). A score's error is that of its
    exponential (a few 2^-24) and of the sum, whose longest chain is E / 64 + 6 terms: less than 2^-19 of it."""
    torch.manual_seed(E + k)
    z = (torch.randn(300, E) * 8).round() / 4
    best = z.view(300, groups, -1).amax(-1)
    shut = torch.ones(300, groups, dtype=torch.bool).scatter_(1, torch.sort(best, descending=True, stable=True).indices[:, :keep], False)
    ranked = z.masked_fill(shut.repeat_interleave(E // groups, 1), float("-inf"))   # (scores are in the order of their logits)
    want_i = torch.sort(ranked, descending=True, stable=True).indices[:, :k]
    want_w = 2.5 * torch.softmax(z.double(), 1).gather(1, want_i)
    eye = torch.eye(E, device=cuda)
    for a, b in ((0, 300), (0, 256), (256, 300)):    # selection alone, fused
        w, i = mix.route_grouped_topk(z[a:b].to(cuda), eye, k, groups, keep, 2.5)
        assert torch.equal(i.cpu().long(), want_i[a:b])
        assert ((w.cpu().double() - want_w[a:b]).abs() <= 2.0 ** -19 * want_w[a:b]).all()


@pytest.mark.parametrize("H", [8, 520, 2056, 4096])
@pytest.mark.parametrize("E", [1, 3, 15, 16, 17, 32, 33, 40, 65, 100])
def test_logits_of_rows_beyond_a_turn(cuda, H, E):
    """A row a wave, sixteen waves, turn after turn: whole turns, one row more or less. (At a width of 4096 routers of 17 - 64 rows go in blocks of 16
    rows on the matrix cores; at the others, no multiples of 64, and with more rows by waves too.)"""
    torch.manual_seed(H + E)
    x, r = torch.randn(5, H, device=cuda).bfloat16(), torch.randn(E, H, device=cuda).bfloat16() / H ** 0.5
    z = x.double() @ r.double().t()
    w, i = mix.route_grouped_topk(x, r, E)
    s = torch.softmax(z, 1).gather(1, i.long())
    # a logit's fp32 sum: H / 64 + 6 additions in a row of 2^-24 of the terms' sum
    e = (H / 64 + 8) * 2.0 ** -24 * float((x.double().abs() @ r.double().abs().t()).max()) + 2.0 ** -20
    assert i.long().sort(1).values.equal(torch.arange(E, device=cuda).expand(5, E)) and ((w.double() - s).abs() <= 3 * e * s).all()
    w, i = mix.route_sigmoid_topk(x, r, E)
    assert i.long().sort(1).values.equal(torch.arange(E, device=cuda).expand(5, E))
    s = torch.sigmoid(z).gather(1, i.long())
    assert ((w.double() - s).abs() <= 3 * e * s).all()


@pytest.mark.parametrize("T,H", [(1, 64), (40, 576), (257, 64), (300, 576), (271, 2048), (513, 4160), (4097, 64), (4130, 128)])
@pytest.mark.parametrize("E,k,groups,keep", [(1, 1, 1, 1), (16, 3, 4, 2), (17, 17, 1, 1), (31, 2, 1, 1), (32, 4, 8, 4), (33, 6, 11, 2), (63, 5, 7, 3), (64, 8, 8, 2)])
def test_prompts_in_rows(cuda, T, H, E, k, groups, keep):
    """Tokens and a router of small whole numbers: logits exact in fp32 in any order of their sum, and full of ties. A score's error is that of
    its exponential (a few 2^-24) and of a sum of at most 64 terms one after the other: less than 2^-17 of it."""
    torch.manual_seed(T + H + E)
    wide = torch.randint(-2, 3, (T, H + 8), device=cuda).bfloat16()
    x, r = wide[:, :H], torch.randint(-2, 3, (E + 1, H), device=cuda).bfloat16()
    z = (x.double() @ r.double().t() / 64).cpu()     # (a 64th: scores stay apart from 0 and 1)
    x = x * 0.125
    x = torch.cat([x, x[:, :8]], 1)[:, :H]           # rows that are no neighbours
    r = r * 0.125

    def check(w, i, score, ranked):
        want = torch.sort(ranked, descending=True, stable=True).indices[:, :k]
        assert torch.equal(i.cpu().long(), want)
        s = score.gather(1, want)
        assert ((w.cpu().double() - s).abs() <= 2.0 ** -17 * s).all()

    z, zg = z[:, :E], z[:, E]
    w, i = mix.route_sigmoid_topk(x, r[:E], k)
    check(w, i, torch.sigmoid(z), z)
    best = z.view(T, groups, -1).amax(-1)
    shut = torch.ones(T, groups, dtype=torch.bool).scatter_(1, torch.sort(best, descending=True, stable=True).indices[:, :keep], False)
    w, i = mix.route_grouped_topk(x, r[:E], k, groups, keep, 2.5)
    check(w, i, 2.5 * torch.softmax(z, 1), z.masked_fill(shut.repeat_interleave(E // groups, 1), float("-inf")))
    for gated in (False, True):
        w, i, g = mix.route_softmax_topk(x, r, k, E, None, gated)
        s = torch.softmax(z, 1)
        top = torch.sort(z, descending=True, stable=True).indices[:, :k]
        check(w, i, s / s.gather(1, top).sum(1, keepdim=True), z)
        assert g is None if not gated else torch.allclose(g.cpu().double(), torch.sigmoid(zg), rtol=2.0 ** -17, atol=0)


@pytest.mark.parametrize("name", ["route_sigmoid_topk", "route_softmax_topk", "route_grouped_topk"])
def test_rows_that_go_to_the_library(cuda, name):
    """Tokens at no multiple of 16 bytes, a router that is not contiguous, fp32 factors, 65 choices, a width of no whole blocks: the same answers."""
    torch.manual_seed(7)
    T, H, E = 300, 192, 20
    x, r = torch.randint(-2, 3, (T, H), device=cuda).bfloat16() / 8, torch.randint(-2, 3, (65, H), device=cuda).bfloat16() / 8

    def go(x, r):
        return (mix.route_softmax_topk(x, r, 3, r.shape[0]) if "softmax" in name else getattr(mix, name)(x, r, 3))[:2]

    odd = torch.empty(T * H + 1, device=cuda, dtype=torch.bfloat16)[1:].view(T, H).copy_(x)
    w, i = go(x, r[:E])
    for a, b in ((odd, r[:E]), (x, r[:E].t().contiguous().t()), (x.float(), r[:E].float())):
        v, j = go(a, b)
        assert torch.equal(i, j) and torch.allclose(w, v, rtol=2.0 ** -17, atol=0)
    for a, b in ((x, r), (x[:, :100].contiguous(), r[:E, :100].contiguous())):
        (v, j), (u, k) = go(a, b), go(a.float(), b.float())
        assert torch.equal(j, k) and torch.allclose(u, v, rtol=2.0 ** -17, atol=0)


@pytest.mark.parametrize("T", [5, 300])
@pytest.mark.parametrize("E", [8, 16, 20, 64, 70])
def test_sigmoid_choice_of_infinite_and_nan_logits(cuda, E, T):
    """Whichever kernel forms the logits: -inf is the smallest of them, each its own choice with weight 0; NaN is none."""
    torch.manual_seed(E + T)
    x, r = torch.randint(1, 4, (T, 128)).bfloat16(), torch.randint(-2, 3, (E, 128)).bfloat16() / 32
    r[2, 5] = r[5, 100] = r[E - 1, 0] = float("-inf")
    w, i = mix.route_sigmoid_topk(x.to(cuda), r.to(cuda), E)
    v, j = mix.route_sigmoid_topk(x, r, E)
    assert torch.equal(i.cpu(), j) and torch.allclose(w.cpu(), v, rtol=2.0 ** -17, atol=0) and (w[:, -3:] == 0).all()
    r[3, 7] = float("nan")
    w, i = mix.route_sigmoid_topk(x.to(cuda), r.to(cuda), E - 1)
    keep = j != 3
    assert torch.equal(i.cpu(), j[keep].view(T, E - 1)) and torch.allclose(w.cpu(), v[keep].view(T, E - 1), rtol=2.0 ** -17, atol=0)


@pytest.mark.parametrize("n,E", [(100, 4), (3000, 16)])
def test_align_leaves_out_what_is_no_expert(cuda, n, E):
    torch.manual_seed(n)
    ids = torch.randint(-1, E + 2, (n,), device=cuda, dtype=torch.int32)
    off, at, pos = (torch.full((s,), -7, dtype=torch.int32, device=cuda) for s in (E + 1, n, n))
    mix._kern().moe_align(off, at, pos, ids, E)
    real = (ids >= 0) & (ids < E)
    m = int(real.sum())
    assert off.tolist() == [0, *torch.bincount(ids[real].long(), minlength=E).cumsum(0).tolist()]
    assert (at[m:] == -7).all() and (pos[~real] == -7).all() and torch.equal(at[pos[real].long()].long(), real.nonzero().flatten())
    assert torch.equal(ids[at[:m].long()], ids[real].sort().values)


@pytest.mark.parametrize("E,h,f,k,kind", [(64, 1024, 512, 2, mix.ACT_CLAMPED), (129, 512, 512, 3, mix.ACT_RELU2), (64, 1024, 576, 2, mix.ACT_SILU)])
def test_experts_of_65_tokens_and_more(cuda, E, h, f, k, kind):
    """Large decode steps go through the grouped product where it tiles (f = 576 it does not), eagerly and replayed: the same as 64 tokens at a time,
    up to rounding. A hidden value is rounded once on one side, on the other with f = 576 three times, of which the gate's may count double (|g| up
    to 3): 2^-9 3^-0.5 (1 + 1 + 4 + 1)^0.5 = 1.5 * 2^-9 root mean square; where both choices are one expert it adds up, 2^0.5 of a result's; 4.5
    sigma (of 10^5 results) are 4.9 * 2^-8. The k experts' results are rounded themselves, 2^-9 each, with weights up to 1.25: 2^-8 k of the
    value and 1.3 * 2^-8 of the root mean square. Where weights scale the input, the 64 tokens' side rounds the scaled row too, which adds (4 + 1) to the
    hidden value's 7: 2 * 2^-9, and with the rest as above 6.4 * 2^-8."""
    torch.manual_seed(E + h)
    T, wide = 128, 2 if kind != mix.ACT_RELU2 else 1
    x = torch.randn(T, h, device=cuda).bfloat16()
    w13, w2 = torch.randn(E, wide * f, h, device=cuda).bfloat16() / h ** 0.5, torch.randn(E, h, f, device=cuda).bfloat16() / f ** 0.5
    ids = torch.randint(0, E + 2, (T, k), device=cuda, dtype=torch.int32)
    w = torch.rand(T, k, device=cuda) + 0.25

    def weighted(a, b):
        return mix.moe_output_weighted(x[a:b], w13, w2, w[a:b], ids[a:b], kind, 1.5, 1.7, E + 2)

    def scaled(a, b):
        return mix.moe_input_scaled(x[a:b], w13, w2, w[a:b], ids[a:b] % E)

    for step in (weighted, scaled) if wide == 2 else (weighted,):
        want = torch.cat([step(0, 64), step(64, T)])
        tol = 2.0 ** -8 * (k * want.abs() + (7.7 if step is scaled else 6.2) * want.square().mean(1, keepdim=True).sqrt())
        for b in (65, 97, T):
            assert ((step(0, b) - want[:b]).abs() <= tol[:b]).all()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            out = step(0, T)
        for _ in range(3):
            out.zero_()
            g.replay()
            assert ((out - want).abs() <= tol).all()
            torch.cuda.synchronize()
