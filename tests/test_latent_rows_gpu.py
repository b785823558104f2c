"""Latent attention of prompt-sized steps: the matrix-core kernel with its queries in registers against the fp32 FMA kernel, at
remainders of its row and key tiles, every rotary width, page sizes that are no power of two and more pages than its table holds.

The matrix-core side rounds softmax weights to bf16 (2^-9 of sum w |v|) and rotated queries (2^-9 of |q| in each of the rot_dim
places: at most e = scale 2^-9 |q_rot| |k_rot| in a score, which moves weights by e^2e); both sides round results (2^-8 each)."""

import pytest
import torch

from src import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rank,rot,heads,bs,window,past", [
    (256, 32, 32, 16, 0, 0), (256, 64, 32, 24, 70, 100), (128, 16, 31, 1, 0, 1200), (64, 0, 32, 7, 0, 50), (256, 0, 33, 16, 33, 300),
    (128, 64, 32, 16, 0, 33), (256, 16, 32, 1, 0, 1100), (64, 32, 32, 48, 200, 0)])
def test_against_fma(cuda, rank, rot, heads, bs, window, past):
    torch.manual_seed(rank + rot + heads)
    S = 72   # with up to 64 tokens each: enough row tiles that the keys are not split
    lens = [64, 1, 33, 2, 63, 31, 17, 48] * (S // 8)
    pasts = [past + 5 * (s % 3) if past else 0 for s in range(S)]
    T, need = sum(lens), [-(-(n + p) // bs) for n, p in zip(lens, pasts)]
    pool = 1 + max(need) * 3
    cache = torch.randn(pool, bs, rank + rot, device=cuda).to(torch.bfloat16)
    bt = torch.randint(0, pool, (S, max(need)), device=cuda, dtype=torch.int32)
    cu = torch.tensor([0] + lens, device=cuda).cumsum(0).int()
    pos = torch.cat([torch.arange(n) + p for n, p in zip(lens, pasts)]).to(cuda)
    ctx = torch.tensor([n + p for n, p in zip(lens, pasts)], device=cuda, dtype=torch.int32)
    q_lat = torch.randn(heads, T, rank, device=cuda).to(torch.bfloat16)
    q = torch.randn(T, heads * (rot + 6), device=cuda).to(torch.bfloat16)
    inv, sink, scale = ops.rope_inv_freq(10000.0, max(rot, 2), cuda)[: rot // 2], torch.randn(heads, device=cuda) + 1, 0.08
    args = (q_lat, q, 6, cache, bt, cu, ctx, pos, sink, 64, window, scale, rot, inv)
    want, got = ops.latent_attn(*args, impl=1).float(), ops.latent_attn(*args, impl=2).float()
    e = 0.0
    if rot:
        e = scale * 2 ** -9 * float(q.view(T, heads, -1)[..., 6:].float().norm(dim=-1).max() * cache[..., rank:].float().norm(dim=-1).max())
    top = float(cache[..., :rank].float().abs().max())
    assert ((got - want).abs() <= (2 ** -9 + 2 * e * 2.71828 ** (2 * e)) * top + 2 ** -7 * want.abs()).all()
    # the bound above is for one key that has it all; over a row the roundings average out
    assert ((got - want).norm() / want.norm()).item() < 2 ** -7


@pytest.mark.parametrize("rank,rot,heads,bs,window,lens,past", [
    (256, 32, 16, 16, 0, (130, 97), 0), (256, 64, 16, 24, 70, (40, 1, 33, 64), 300), (128, 16, 33, 1, 0, (31, 12), 1200), (64, 0, 20, 7, 33, (60,) * 8, 50),
    (256, 0, 5, 16, 0, (100, 64, 7), 40), (256, 16, 32, 16, 0, (16,) * 8, 90)])
def test_few_row_tiles(cuda, rank, rot, heads, bs, window, lens, past):
    """32 rows per wave, two waves to a row's value columns: steps of up to two workgroups per compute unit, unsplit."""
    from src.ops import mix

    torch.manual_seed(rank + rot + heads)
    S, T, need = len(lens), sum(lens), -(-(max(lens) + past) // bs)
    cache = torch.randn(1 + 3 * need, bs, rank + rot, device=cuda).to(torch.bfloat16)
    bt = torch.randint(0, 1 + 3 * need, (S, need), device=cuda, dtype=torch.int32)
    cu = torch.tensor([0, *lens], device=cuda).cumsum(0).int()
    pos = torch.cat([torch.arange(n) + past for n in lens]).to(cuda)
    ctx = torch.tensor([n + past for n in lens], device=cuda, dtype=torch.int32)
    q_lat = torch.randn(heads, T, rank, device=cuda).to(torch.bfloat16)
    q = torch.randn(T, heads * (rot + 6), device=cuda).to(torch.bfloat16)
    inv, sink, scale = ops.rope_inv_freq(10000.0, max(rot, 2), cuda)[: rot // 2], torch.randn(heads, device=cuda) + 1, 0.08
    got = torch.empty_like(q_lat)
    tail = (cache, bt, cu, ctx, pos, sink, max(lens), window, scale, rot, inv)
    form = mix._kern().latent_attn_named(got, q_lat, q, 6, *tail, 0)
    assert form == ("split" if past >= 1000 else "wide")   # (few rows behind that many keys)
    want = ops.latent_attn(q_lat, q, 6, *tail, impl=1).float()
    e = 0.0
    if rot:
        e = scale * 2 ** -9 * float(q.view(T, heads, -1)[..., 6:].float().norm(dim=-1).max() * cache[..., rank:].float().norm(dim=-1).max())
    top = float(cache[..., :rank].float().abs().max())
    assert ((got.float() - want).abs() <= (2 ** -9 + 2 * e * 2.71828 ** (2 * e)) * top + 2 ** -7 * want.abs()).all()
    assert ((got.float() - want).norm() / want.norm()).item() < 2 ** -7


@pytest.mark.parametrize("rank,rot,heads,bs,lens,past,kernel", [
    (256, 32, 16, 1, (1300,), 0, "wide"), (256, 16, 16, 24, (1300,), 0, "wide"), (64, 0, 12, 16, (700, 600), 700, "wide"), (128, 64, 16, 7, (1100,), 60, "wide"),
    (256, 32, 16, 1, (1100, 1100), 0, "rows")])
def test_row_table_is_filled_again(cuda, rank, rot, heads, bs, lens, past, kernel):
    """More visible keys than the 1024 entries that a workgroup's table holds, at page sizes of 1 and others."""
    from src.ops import mix

    torch.manual_seed(rank + rot + bs)
    S, T, need = len(lens), sum(lens), -(-(max(lens) + past) // bs)
    cache = torch.randn(1 + 2 * need, bs, rank + rot, device=cuda).to(torch.bfloat16)
    bt = torch.randint(0, 1 + 2 * need, (S, need), device=cuda, dtype=torch.int32)
    cu = torch.tensor([0, *lens], device=cuda).cumsum(0).int()
    pos = torch.cat([torch.arange(n) + past for n in lens]).to(cuda)
    ctx = torch.tensor([n + past for n in lens], device=cuda, dtype=torch.int32)
    q_lat, q = torch.randn(heads, T, rank, device=cuda).to(torch.bfloat16), torch.randn(T, heads * (rot + 6), device=cuda).to(torch.bfloat16)
    inv, sink, scale = ops.rope_inv_freq(10000.0, max(rot, 2), cuda)[: rot // 2], torch.randn(heads, device=cuda) + 1, 0.08
    got = torch.empty_like(q_lat)
    tail = (cache, bt, cu, ctx, pos, sink, max(lens), 0, scale, rot, inv)
    assert mix._kern().latent_attn_named(got, q_lat, q, 6, *tail, 0) == kernel
    want = ops.latent_attn(q_lat, q, 6, *tail, impl=1).float()
    e = 0.0
    if rot:
        e = scale * 2 ** -9 * float(q.view(T, heads, -1)[..., 6:].float().norm(dim=-1).max() * cache[..., rank:].float().norm(dim=-1).max())
    top = float(cache[..., :rank].float().abs().max())
    assert ((got.float() - want).abs() <= (2 ** -9 + 2 * e * 2.71828 ** (2 * e)) * top + 2 ** -7 * want.abs()).all()
    assert ((got.float() - want).norm() / want.norm()).item() < 2 ** -7


@pytest.mark.parametrize("rot,heads,bs,window,lens,past,kernel", [
    (32, 32, 16, 0, (520, 511, 497, 520, 33, 519, 520, 512, 520), 0, "two rows"), (16, 31, 24, 300, (600, 590, 1, 600, 600, 130, 600), 200, "two rows"),
    (0, 33, 7, 0, (700, 655, 700, 690, 129), 300, "two rows"), (64, 32, 1, 0, (650,) * 5, 1000, "two rows"), (32, 16, 1, 0, (1400, 1400), 0, "two rows"),
    (32, 32, 16, 0, (250, 130) * 4, 0, "rows")])
def test_two_groups_of_rows(cuda, rot, heads, bs, window, lens, past, kernel):
    """Two groups of 16 rows per wave: remainders of the workgroups' 128 rows and of key tiles, windows, every rotary width, the table filled again."""
    from src.ops import mix

    rank = 256
    torch.manual_seed(rot + heads + bs)
    S, T, need = len(lens), sum(lens), -(-(max(lens) + past) // bs)
    cache = torch.randn(1 + 2 * need, bs, rank + rot, device=cuda).to(torch.bfloat16)
    bt = torch.randint(0, 1 + 2 * need, (S, need), device=cuda, dtype=torch.int32)
    cu = torch.tensor([0, *lens], device=cuda).cumsum(0).int()
    pos = torch.cat([torch.arange(n) + past for n in lens]).to(cuda)
    ctx = torch.tensor([n + past for n in lens], device=cuda, dtype=torch.int32)
    q_lat, q = torch.randn(heads, T, rank, device=cuda).to(torch.bfloat16), torch.randn(T, heads * (rot + 6), device=cuda).to(torch.bfloat16)
    inv, sink, scale = ops.rope_inv_freq(10000.0, max(rot, 2), cuda)[: rot // 2], torch.randn(heads, device=cuda) + 1, 0.08
    got = torch.empty_like(q_lat)
    tail = (cache, bt, cu, ctx, pos, sink, max(lens), window, scale, rot, inv)
    assert mix._kern().latent_attn_named(got, q_lat, q, 6, *tail, 0) == kernel
    want = ops.latent_attn(q_lat, q, 6, *tail, impl=1).float()
    e = 0.0
    if rot:
        e = scale * 2 ** -9 * float(q.view(T, heads, -1)[..., 6:].float().norm(dim=-1).max() * cache[..., rank:].float().norm(dim=-1).max())
    top = float(cache[..., :rank].float().abs().max())
    assert ((got.float() - want).abs() <= (2 ** -9 + 2 * e * 2.71828 ** (2 * e)) * top + 2 ** -7 * want.abs()).all()
    assert ((got.float() - want).norm() / want.norm()).item() < 2 ** -7


def test_results_at_any_8_bytes(cuda):
    """Results that start at no multiple of 16 bytes go to the kernel that writes 8 at a time: the bits that it writes anywhere."""
    from src.ops import mix

    torch.manual_seed(3)
    S, n, heads, rank, rot = 64, 40, 32, 64, 16
    T, pages = S * n, 3
    cache = torch.randn(S * pages, 16, rank + rot, device=cuda).to(torch.bfloat16)
    bt = torch.randperm(S * pages, device=cuda).int().view(S, pages)
    cu = (torch.arange(S + 1, device=cuda) * n).int()
    pos, ctx = torch.arange(n, device=cuda).repeat(S), torch.full((S,), n, device=cuda, dtype=torch.int32)
    q_lat, q = torch.randn(heads, T, rank, device=cuda).to(torch.bfloat16), torch.randn(T, heads * rot, device=cuda).to(torch.bfloat16)
    room = torch.zeros(heads * T * rank + 8, device=cuda, dtype=torch.bfloat16)

    def at(start, impl):
        out = room[start:start + heads * T * rank].view(heads, T, rank)
        form = mix._kern().latent_attn(out, q_lat, q, 0, cache, bt, cu, ctx, pos, None, n, 0, 0.1, rot, ops.rope_inv_freq(1e4, rot, cuda), impl)
        return form, out.clone()

    form, want = at(0, 3)
    assert form == "tiles" and at(0, 0)[0] == "rows"
    form, got = at(4, 0)
    assert form == "tiles" and torch.equal(got, want)


@pytest.mark.parametrize("lens,window", [((64, 1, 33, 2, 63, 31, 17, 48) * 8 + (5, 64, 9), 0), ((200, 333, 1, 140, 257, 90, 310, 16, 128), 70),
                                         ((70, 2, 55, 64, 9, 33, 70, 41) * 2, 0), ((199, 101, 1, 160, 177, 200, 140, 33) * 3, 0), ((5, 64, 1, 17, 32, 40, 63, 2) * 4, 0)])
def test_sequences_not_in_eights(cuda, lens, window):
    """The row tiles of a number of sequences that is no multiple of 8, or a small one of unequal lengths, are dealt in another order: every
    row once, the longest sequence's too."""
    torch.manual_seed(len(lens))
    rank, rot, heads, bs, scale = 256, 32, 32, 16, 0.08
    S, T, need = len(lens), sum(lens), -(-max(lens) // bs)
    cache = torch.randn(1 + 3 * need, bs, rank + rot, device=cuda).to(torch.bfloat16)
    bt = torch.randint(0, 1 + 3 * need, (S, need), device=cuda, dtype=torch.int32)
    cu = torch.tensor([0, *lens], device=cuda).cumsum(0).int()
    pos = torch.cat([torch.arange(n) for n in lens]).to(cuda)
    ctx = torch.tensor(lens, device=cuda, dtype=torch.int32)
    q_lat = torch.randn(heads, T, rank, device=cuda).to(torch.bfloat16)
    q = torch.randn(T, heads * (rot + 6), device=cuda).to(torch.bfloat16)
    inv, sink = ops.rope_inv_freq(10000.0, rot, cuda)[: rot // 2], torch.randn(heads, device=cuda) + 1
    args = (q_lat, q, 6, cache, bt, cu, ctx, pos, sink, max(lens), window, scale, rot, inv)
    want, got = ops.latent_attn(*args, impl=1).float(), ops.latent_attn(*args).float()
    e = scale * 2 ** -9 * float(q.view(T, heads, -1)[..., 6:].float().norm(dim=-1).max() * cache[..., rank:].float().norm(dim=-1).max())
    top = float(cache[..., :rank].float().abs().max())
    assert ((got - want).abs() <= (2 ** -9 + 2 * e * 2.71828 ** (2 * e)) * top + 2 ** -7 * want.abs()).all()
    assert ((got - want).norm() / want.norm()).item() < 2 ** -7
