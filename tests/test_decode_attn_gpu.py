"""Decode attention (one bf16 query row per sequence): the wave-per-keys kernel against the plain form, around the sizes where
its waves, trips and splits begin and end. Scores, weights and sums are fp32 on both sides; results are rounded to bf16, where two
sums that differ in their last bits may round to different neighbours (2^-7 of the value at most; 1e-4 of the largest for values
that cancel)."""

import pytest
import torch

from src.ops import seq

pytestmark = pytest.mark.gpu
CTX = [1, 2, 15, 16, 17, 31, 33, 64, 65, 127, 128, 129, 160, 257, 513, 1000]


def _case(dim, vdim, heads, groups, bs, width):
    S, n = len(CTX), sum(-(-c // bs) for c in CTX)
    cache = torch.randn(n + 1, bs, groups * (dim + vdim)).to(torch.bfloat16)
    ids, bt = torch.randperm(n) + 1, torch.zeros(S, width // bs + 1, dtype=torch.int32)
    for s, c in enumerate(CTX):
        k = -(-c // bs)
        bt[s, :k], ids = ids[:k].int(), ids[k:]
    return torch.randn(S, heads * dim).to(torch.bfloat16), cache, bt, torch.tensor(CTX, dtype=torch.int32), torch.tensor(CTX) - 1


@pytest.mark.parametrize("dim,vdim,heads,groups,bs,style", [
    (128, 128, 8, 2, 16, ""), (128, 128, 6, 2, 16, "sink"), (64, 64, 16, 2, 16, "cap"), (72, 40, 2, 2, 16, "bias"), (8, 8, 2, 1, 16, "sink"),
    (256, 256, 8, 1, 16, ""), (192, 128, 4, 2, 32, "sigmoid"), (128, 256, 4, 1, 16, "window"), (64, 128, 5, 1, 24, "sink"),
    (96, 96, 4, 4, 64, "seg"), (128, 128, 2, 2, 16, "sigmoid"), (256, 64, 6, 2, 8, "window")])
@pytest.mark.parametrize("width", [1000, 16000])   # the block table's width sets the splits: many of them, and empty ones
def test_edges(cuda, dim, vdim, heads, groups, bs, style, width):
    torch.manual_seed(dim + vdim + heads)
    q, cache, bt, ctx, pos = _case(dim, vdim, heads, groups, bs, width)
    sink, bias, window, kw = None, None, 0, {}
    if style == "sink":
        sink = torch.randn(heads) + 2
    if style == "bias":
        sink, bias = torch.randn(heads), torch.randn(40, heads)
    if style == "cap":
        kw = dict(softcap=5.0, slopes=torch.rand(heads) * 0.1)
    if style == "sigmoid":
        kw = dict(sigmoid=True, head_bias=torch.randn(heads) - 3)
    if style == "seg":
        kw = dict(seg=100)
    if style == "window":
        window = 130
    args = lambda dev: [t if t is None else t.to(dev) for t in (q, cache, bt, None, ctx, pos, sink, bias)]
    put = lambda dev: {k: v.to(dev) if torch.is_tensor(v) else v for k, v in kw.items()}
    want = seq.sink_attn(*args("cpu"), 1, heads, groups, dim, vdim, window, dim ** -0.5, **put("cpu")).float()
    got = seq.sink_attn(*args(cuda), 1, heads, groups, dim, vdim, window, dim ** -0.5, **put(cuda)).float().cpu()
    assert ((got - want).abs() <= 2 ** -7 * want.abs() + 1e-4 * want.abs().max()).all()


def test_cache_of_more_rows_than_32_bits_count(cuda):
    """The narrowest rows (8 + 8 values): blocks on either side of row 2^32 of one cache. Rows counted in 32 bits would be those of
    the first blocks, which hold other values."""
    bs, high = 16, 2 ** 28   # block 2^28 starts at row 2^32
    if torch.cuda.mem_get_info()[0] < 160 * 2 ** 30:
        pytest.skip("the cache takes 128 GiB")
    torch.manual_seed(0)
    heads, dim, vdim, ctx = 2, 8, 8, torch.tensor([90, 33], dtype=torch.int32)
    small = torch.randn(16, bs, dim + vdim).to(torch.bfloat16)
    big = torch.empty(high + 8, bs, dim + vdim, dtype=torch.bfloat16, device=cuda)
    big[:8] = 9.0
    big[high - 8:] = small.to(cuda)
    near = torch.tensor([[7, 8, 15, 3, 10, 9], [12, 0, 8, 1, 2, 4]], dtype=torch.int32)
    q = torch.randn(2, heads * dim).to(torch.bfloat16)
    pos = ctx.long() - 1
    want = seq.sink_attn(q, small, near, None, ctx, pos, None, None, 1, heads, 1, dim, vdim, 0, 0.35).float()
    got = seq.sink_attn(q.to(cuda), big, (near + high - 8).to(cuda), None, ctx.to(cuda), pos.to(cuda), None, None, 1, heads, 1, dim, vdim,
                        0, 0.35).float().cpu()
    del big
    torch.cuda.empty_cache()
    assert ((got - want).abs() <= 2 ** -7 * want.abs() + 1e-4 * want.abs().max()).all()
