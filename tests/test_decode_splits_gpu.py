"""Attention of decode steps whose splits take trips of 128 keys in turn: numbers of workgroups that go in one, three, five and many splits,
sequences shorter than one trip of all splits, tables far wider than any sequence, against the fp32 FMA kernel.

Scores of bf16 rows are exact products summed in fp32, weights and sums are fp32 on both sides (some 2^-20 of the largest value), results are
rounded to bf16 on both (2^-8 of a value in all)."""

import pytest
import torch

from src.ops import seq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,G,rep,dim,vdim,longest,wide,kw", [
    (36, 8, 2, 64, 64, 700, 0, {}), (70, 8, 1, 64, 64, 500, 0, {}), (3, 2, 4, 128, 128, 1500, 100, {}), (64, 8, 1, 64, 128, 300, 0, {}), (5, 4, 8, 128, 256, 900, 0, {}),
    (40, 8, 2, 64, 64, 400, 300, {"window": 200}), (2, 4, 2, 128, 128, 129, 0, {"sink": True}), (37, 8, 2, 64, 64, 260, 0, {"sigmoid": True})])
def test_splits_in_turn(cuda, S, G, rep, dim, vdim, longest, wide, kw):
    torch.manual_seed(S + G + longest)
    H = G * rep
    ctx = torch.tensor([1 + (i * 37) % longest if i else longest for i in range(S)], dtype=torch.int32, device=cuda)
    need = -(-longest // 16) + wide
    bt = torch.randint(0, 400, (S, need), device=cuda, dtype=torch.int32)
    cache, q = torch.randn(400, 16, G * (dim + vdim), device=cuda).bfloat16(), torch.randn(S, H * dim, device=cuda).bfloat16()
    sink = torch.randn(H, device=cuda) if kw.get("sink") else None
    ext = {"sigmoid": True} if kw.get("sigmoid") else {}
    args = (q, cache, bt, None, ctx, (ctx - 1).long(), sink, None, 1, H, G, dim, vdim, kw.get("window", 0), dim ** -0.5)
    got, want = seq.sink_attn(*args, **ext).float(), seq.sink_attn(*args, impl=1, **ext).float()
    assert ((got - want).abs() <= 2 ** -7 * want.abs() + 2 ** -16 * want.abs().max()).all()
