"""Latent attention of decode steps: the kernel whose waves own their keys against the fp32 FMA kernel, over tile remainders, head blocks,
rotary widths, pages that are no power of two, windows, splits that hold nothing and a captured step.

The matrix-core side rounds softmax weights to bf16 (2^-9 of sum w |v|) and rotated queries (2^-9 of |q| in each of the rot_dim
places: at most e = scale 2^-9 |q_rot| |k_rot| in a score, which moves weights by e^2e); both sides round results (2^-8 each)."""

import pytest
import torch

from src import ops
from src.ops import mix

pytestmark = pytest.mark.gpu


def _case(cuda, rank, rot, heads, bs, ctxs, wide=0):
    torch.manual_seed(rank + rot + heads + bs)
    S, need = len(ctxs), -(-max(ctxs) // bs) + wide
    cache = torch.randn(1 + 2 * need, bs, rank + rot, device=cuda).to(torch.bfloat16)
    bt = torch.randint(0, 1 + 2 * need, (S, need), device=cuda, dtype=torch.int32)
    ctx = torch.tensor(ctxs, device=cuda, dtype=torch.int32)
    q_lat = torch.randn(heads, S, rank, device=cuda).to(torch.bfloat16)
    q = torch.randn(S, heads * (rot + 6), device=cuda).to(torch.bfloat16)
    inv = ops.rope_inv_freq(10000.0, max(rot, 2), cuda)[: rot // 2]
    return q_lat, q, 6, cache, bt, None, ctx, (ctx - 1).long(), torch.randn(heads, device=cuda) + 1, 1, 0, 0.08, rot, inv


def _close(got, want, q, cache, rank, rot, heads):
    e = 0.0
    if rot:
        e = 0.08 * 2 ** -9 * float(q.view(q.shape[0], heads, -1)[..., 6:].float().norm(dim=-1).max() * cache[..., rank:].float().norm(dim=-1).max())
    top = float(cache[..., :rank].float().abs().max())
    assert ((got.float() - want).abs() <= (2 ** -9 + 2 * e * 2.71828 ** (2 * e)) * top + 2 ** -7 * want.abs()).all()
    assert ((got.float() - want).norm() / want.norm()).item() < 2 ** -7


@pytest.mark.parametrize("rank,rot,heads,bs,ctxs,window,wide", [
    (256, 32, 16, 16, [1, 31, 32, 33, 128, 129, 700], 0, 0), (256, 64, 33, 24, [900, 5], 70, 0), (128, 16, 5, 1, [64, 2000], 0, 0), (64, 0, 40, 7, [300] * 9, 33, 0),
    (256, 16, 32, 16, [17] * 70, 0, 0), (64, 32, 16, 48, [1500], 0, 60), (128, 64, 17, 16, [640, 1, 96], 0, 200)])
def test_against_fma(cuda, rank, rot, heads, bs, ctxs, window, wide):
    args = list(_case(cuda, rank, rot, heads, bs, ctxs, wide))
    args[10] = window
    got = torch.empty_like(args[0])
    assert mix._kern().latent_attn_named(got, *args, 0) == "decode"
    _close(got, ops.latent_attn(*args, impl=1).float(), args[1], args[3], rank, rot, heads)
    args[8] = None   # without a sink
    _close(ops.latent_attn(*args), ops.latent_attn(*args, impl=1).float(), args[1], args[3], rank, rot, heads)


def test_captured_step_follows_its_lengths(cuda):
    """A step is captured with tables as wide as the longest sequence may be, and replayed at other lengths."""
    args = _case(cuda, 256, 32, 16, 16, [1, 1, 1, 1], 64)
    ctx, pos = args[6], args[7]
    ops.latent_attn(*args)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.latent_attn(*args)
    for lens in ([5, 900, 32, 1], [1000, 3, 128, 640], [1, 1, 1, 1], [1000, 1000, 999, 1000]):
        ctx.copy_(torch.tensor(lens, dtype=torch.int32))
        pos.copy_(ctx - 1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ops.latent_attn(*args))
        _close(out, ops.latent_attn(*args, impl=1).float(), args[1], args[3], 256, 32, 16)


@pytest.mark.parametrize("rank,heads,scale", [(256, 40, 0.15), (128, 64, 0.2), (64, 128, 0.3)])
@pytest.mark.parametrize("ctxs", [[60, 100, 33], [700, 40]])
def test_weights_of_many_heads_keep_16_bits(cuda, rank, heads, scale, ctxs):
    """More than 32 heads: two bf16 parts of the weights. What they leave (2^-17) is nothing beside the results' own rounding, whose distance from
    64 bits a correct kernel therefore has; one part (2^-9 of each weight, few keys carrying most of the sum) adds 5 % and more to it."""
    args = list(_case(cuda, rank, 0, heads, 16, ctxs))
    args[11] = scale
    got = ops.latent_attn(*args)
    q, cache, bt, ctx, sink = args[0].double(), args[3].double(), args[4].long(), args[6].tolist(), args[8].double()
    want = torch.empty_like(q)
    for s, n in enumerate(ctx):
        rows = cache[bt[s]].reshape(-1, rank)[:n]
        sc = torch.cat([q[:, s] @ rows.t().contiguous() * scale, sink[:, None]], 1)
        want[:, s] = torch.softmax(sc, 1)[:, :n] @ rows
    assert (got.double() - want).norm() <= 1.01 * (want.bfloat16().double() - want).norm()
