"""The grouped expert product of prompt-sized steps (moe_gemm.hip) against the same product in float64.

Results are rounded to bf16 once (2^-9 of each value); the fp32 sums of up to 1024 products add about 1024^0.5 * 2^-24 of their
terms' size, which matters only beside cancelled values: 2^-8 of the value plus 2^-8 of the row's root mean square covers both, and
is far below what one wrong row, column or stage moves."""

import pytest
import torch
import torch.nn.functional as F

from src.ops import mix

pytestmark = pytest.mark.gpu


def _case(counts, K, ncols, gated, topk, seed=0):
    """Rows sorted by expert with the given rows per expert; row j reads token sorted[j] / topk."""
    g = torch.Generator().manual_seed(seed)
    n, E = sum(counts), len(counts)
    x = torch.randn(n // topk, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(E, ncols * (2 if gated else 1), K, generator=g) * K ** -0.5).to(torch.bfloat16)
    offsets = torch.tensor([0] + list(counts)).cumsum(0).int()
    return x, w, offsets, torch.randperm(n, generator=g).int(), torch.rand(n, generator=g) + 0.5


def _want(x, w, offsets, idx, topk, act, scale, limit, alpha):
    rows = x.double()[idx.long() // topk] if idx is not None else x.double()
    out = []
    for e in range(w.shape[0]):
        a, b = int(offsets[e]), int(offsets[e + 1])
        z = rows[a:b] @ w[e].double().t()
        if scale is not None:
            z = z * scale.double()[idx[a:b].long()][:, None]
        if act in (mix.MOE_SILU, mix.MOE_CLAMPED, mix.MOE_GELU):
            g, u = z.chunk(2, 1)
            if act == mix.MOE_SILU:
                z = F.silu(g) * u
            elif act == mix.MOE_GELU:
                z = F.gelu(g, approximate="tanh") * u
            else:
                g = g.clamp(max=limit)
                z = g * torch.sigmoid(alpha * g) * (u.clamp(-limit, limit) + 1)
        elif act == mix.MOE_RELU2:
            z = torch.relu(z) ** 2
        out.append(z)
    return torch.cat(out)


# rows per expert: none, one, around a 32-row piece, around a tile of 128 and of 192 - 256 rows, uneven heights, an odd sum
COUNTS = [(0, 1, 31, 32), (33, 0, 95, 64), (129, 127, 0, 256), (257, 255, 193, 63), (700, 0, 0, 4), (65, 0, 97, 3)]


@pytest.mark.parametrize("counts", COUNTS)
@pytest.mark.parametrize("K,ncols,act", [(64, 256, mix.MOE_NONE), (128, 128, mix.MOE_SILU), (192, 256, mix.MOE_CLAMPED),
                                         (1024, 512, mix.MOE_RELU2), (64, 384, mix.MOE_GELU)])
def test_products(cuda, counts, K, ncols, act):
    topk = 2 if sum(counts) % 2 == 0 else 1
    x, w, offsets, idx, scale = _case(counts, K, ncols, act in (mix.MOE_SILU, mix.MOE_CLAMPED, mix.MOE_GELU), topk)
    kern = mix._kern()
    for rows, sc in ((idx, None), (idx, scale), (None, None)):
        xs = x if rows is not None else x.repeat_interleave(topk, 0)
        out = torch.full((sum(counts), ncols), 7.0, dtype=torch.bfloat16, device=cuda)
        dev = [None if t is None else t.to(cuda) for t in (xs, w, offsets, rows, sc)]
        assert kern.moe_gemm(out, *dev[:4], topk if rows is not None else 1, dev[4], act, 1.5, 1.7)
        want = _want(xs, w, offsets, rows, topk, act, sc, 1.5, 1.7)
        tol = 2.0 ** -8 * (want.abs() + want.square().mean(1, keepdim=True).sqrt())
        bad = ((out.cpu().double() - want).abs() > tol).nonzero()
        assert not len(bad), (len(bad), bad[:4].tolist())


@pytest.mark.parametrize("act,kind", [(mix.MOE_SILU, mix.ACT_SILU), (mix.MOE_CLAMPED, mix.ACT_CLAMPED), (mix.MOE_GELU, mix.ACT_GELU_TANH)])
def test_activations_are_those_of_the_separate_pass(cuda, act, kind):
    """Rows with a single one: the sums are the weights themselves, exactly, and the results those of gated_act on the scaled fp32
    values, rounded, to the bf16 value (a million of them, of which a coarser exponential rounds some dozens to the other neighbour)."""
    g = torch.Generator().manual_seed(7)
    n, ncols, K = 8192, 128, 64
    x = torch.zeros(n, K)
    at = torch.randint(0, K, (n,), generator=g)
    x[torch.arange(n), at] = 1.0
    w = (torch.randn(1, 2 * ncols, K, generator=g) * 3).to(torch.bfloat16)
    scale = torch.rand(n, generator=g) + 0.5
    want = mix.gated_act((w[0].float().t()[at] * scale[:, None]).to(cuda), kind, 7.0, 1.702).to(torch.bfloat16)
    out = torch.empty(n, ncols, dtype=torch.bfloat16, device=cuda)
    offsets = torch.tensor([0, n], dtype=torch.int32)
    dev = [t.to(cuda) for t in (x.to(torch.bfloat16), w, offsets)]
    assert mix._kern().moe_gemm(out, *dev, None, 1, scale.to(cuda), act, 7.0, 1.702)
    assert torch.equal(out, want), (out != want).sum()


@pytest.mark.parametrize("height", [128, 160, 192, 224, 256])
@pytest.mark.parametrize("K,ncols,act", [(64, 256, mix.MOE_NONE), (320, 128, mix.MOE_SILU)])
def test_every_tile_height(cuda, height, K, ncols, act):
    """The heights that large steps take, asked for: full tiles, last tiles of one row, around 32 rows and one short of full, several
    tiles of an expert (two waves share a tile's 32-row pieces: 4 and 4, 4 and 3, 3 and 3, 3 and 2, 2 and 2 of them, and all fewer)."""
    counts = (height, height - 1, 1, 31, 33, height + 1, 2 * height + 33, 3 * height, 95, 161)
    x, w, offsets, idx, scale = _case(counts, K, ncols, act != mix.MOE_NONE, 1, seed=height)
    out = torch.full((sum(counts), ncols), 7.0, dtype=torch.bfloat16, device=cuda)
    dev = [t.to(cuda) for t in (x, w, offsets, idx, scale)]
    assert mix._kern().moe_gemm(out, *dev[:4], 1, dev[4], act, 1.5, 1.7, height)
    want = _want(x, w, offsets, idx, 1, act, scale, 1.5, 1.7)
    tol = 2.0 ** -8 * (want.abs() + want.square().mean(1, keepdim=True).sqrt())
    assert ((out.cpu().double() - want).abs() <= tol).all()


@pytest.mark.parametrize("counts", [(475,) * 4, (1024, 0, 3, 900, 511, 513), (97,) * 3 + (600,), (449, 448, 447, 1)])
def test_chosen_heights(cuda, counts):
    """The height that the kernel takes by itself: the same bits as with each of the heights (a row's sums do not depend on its tile)."""
    x, w, offsets, idx, scale = _case(counts, 128, 1024, True, 1, seed=len(counts))
    dev = [t.to(cuda) for t in (x, w, offsets, idx)]
    outs = [torch.full((sum(counts), 1024), 7.0, dtype=torch.bfloat16, device=cuda) for _ in range(6)]
    for out, height in zip(outs, (0, 128, 160, 192, 224, 256)):
        assert mix._kern().moe_gemm(out, *dev, 1, scale.to(cuda), mix.MOE_SILU, 0.0, 0.0, height)
    assert all(torch.equal(outs[0], o) for o in outs[1:])


@pytest.mark.parametrize("counts,K,ncols,act", [
    ((2300, 40, 0, 1900), 64, 512, mix.MOE_NONE),              # more than 8 tiles of an expert share a weight tile
    ((5, 0, 64) * 30, 128, 256, mix.MOE_RELU2),                # more experts than lanes, no full turn of the compute units
    ((300,) * 16, 192, 1024, mix.MOE_SILU),                    # a rest that is cut by rows
    ((2100, 2050, 1990, 2060), 64, 1280, mix.MOE_NONE),        # full turns and a rest; one stage: its successor is another tile's
])
def test_tiles_and_turns(cuda, counts, K, ncols, act):
    x, w, offsets, idx, scale = _case(counts, K, ncols, act == mix.MOE_SILU, 1, seed=K)
    out = torch.full((sum(counts), ncols), 7.0, dtype=torch.bfloat16, device=cuda)
    dev = [t.to(cuda) for t in (x, w, offsets, idx, scale)]
    assert mix._kern().moe_gemm(out, *dev[:4], 1, dev[4], act, 1.5, 1.7)
    want = _want(x, w, offsets, idx, 1, act, scale, 1.5, 1.7)
    tol = 2.0 ** -8 * (want.abs() + want.square().mean(1, keepdim=True).sqrt())
    assert ((out.cpu().double() - want).abs() <= tol).all()


def test_extra_groups_are_left_alone(cuda):
    """Rows behind the last expert (identity entries, other ranks' experts) are not written."""
    x, w, offsets, idx, _ = _case((40, 60), 128, 256, False, 1)
    out = torch.full((100, 256), 3.0, dtype=torch.bfloat16, device=cuda)
    assert mix._kern().moe_gemm(out, x.to(cuda), w[:1].contiguous().to(cuda), offsets.to(cuda), idx.to(cuda), 1, None, mix.MOE_NONE, 0.0, 0.0)
    assert (out[40:] == 3.0).all() and not (out[:40] == 3.0).all()


def test_sizes_that_do_not_tile_are_left_to_the_caller(cuda):
    x, w, offsets, idx, _ = _case((40, 60), 96, 256, False, 1)
    out = torch.empty(100, 256, dtype=torch.bfloat16, device=cuda)
    assert not mix._kern().moe_gemm(out, x.to(cuda), w.to(cuda), offsets.to(cuda), idx.to(cuda), 1, None, mix.MOE_NONE, 0.0, 0.0)


@pytest.mark.parametrize("t,h,f,e,k", [(300, 256, 512, 4, 2), (300, 256, 320, 4, 2), (700, 512, 256, 6, 3)])
def test_mixtures_of_prompt_steps(cuda, t, h, f, e, k):
    """The three mixtures end to end, widths that the grouped product tiles and that it leaves (f = 320: not 256-wide columns)."""
    g = torch.Generator().manual_seed(t + f)
    bf = torch.bfloat16
    x = torch.randn(t, h, generator=g).to(bf)
    w13, w1, w2 = ((torch.randn(*s, generator=g) * 0.05).to(bf) for s in ((e, 2 * f, h), (e, f, h), (e, h, f)))
    ids = torch.rand(t, e + 1, generator=g).argsort(1)[:, :k].int()   # e: an identity entry
    w = torch.rand(t, k, generator=g)
    real = ids.clamp(max=e - 1)
    from src import ops
    from src.ops import reference as ref

    for name, got, want in (
            ("scaled", lambda d: mix.moe_input_scaled(*d(x, w13, w2, w, real)), ref.moe_input_scaled(x, w13, w2, w, real, None)),
            ("weighted", lambda d: mix.moe_output_weighted(*d(x, w13, w2, w, ids), mix.ACT_CLAMPED, 7.0, 1.7, n_route=e + 1),
             ref.moe_output_weighted(x, w13, w2, w, ids, mix.ACT_CLAMPED, 7.0, 1.7, None, None)),
            ("relu2", lambda d: mix.moe_output_weighted(*d(x, w1, w2, w, real), mix.ACT_RELU2, 0.0, 0.0),
             ref.moe_output_weighted(x, w1, w2, w, real, mix.ACT_RELU2, 0.0, 0.0, None, None)),
            ("mixtral", lambda d: ops.moe_apply(*d(x, w13, w2, w, real), e), ref.moe_experts(x, w13, w2, w, real))):
        y = got(lambda *ts: [v.to(cuda) for v in ts]).float().cpu()
        err = (y - want.float()).norm() / want.float().norm()
        assert err < 1e-2, (name, err)   # two roundings to bf16 on either side


@pytest.mark.parametrize("stack", ["slice", "transposed"])
def test_strided_weights_take_the_library(cuda, stack):
    """Expert weights that are views (every other expert of a stack, a wider stack's columns, transposed storage) give the bits of the
    library products on copies of them that the grouped product does not take either (an unaligned start)."""
    from src import ops

    g = torch.Generator().manual_seed(3)
    t, h, f, e, k, bf = 300, 256, 512, 4, 2, torch.bfloat16
    randn = lambda *s: (torch.randn(*s, generator=g) * 0.05).to(bf).to(cuda)
    if stack == "slice":
        w13, w1, w2 = randn(2 * e, 2 * f, h)[::2], randn(e, f, h + 64)[:, :, :h], randn(e, h + 8, f)[:, :h]
    else:
        w13, w1, w2 = (randn(e, h, n).transpose(1, 2) for n in (2 * f, f, f))
        w2 = randn(e, f, h).transpose(1, 2)
    assert not (w13.is_contiguous() or w1.is_contiguous() or w2.is_contiguous())

    def off(v):   # the same values from an address that is no multiple of 16 bytes
        return torch.empty(v.numel() + 1, dtype=bf, device=cuda)[1:].view(v.shape).copy_(v)

    x, w = torch.randn(t, h, generator=g).to(bf).to(cuda), torch.rand(t, k, generator=g).to(cuda)
    ids = torch.rand(t, e, generator=g).argsort(1)[:, :k].int().to(cuda)
    for run in (lambda a, _, c: mix.moe_input_scaled(x, a, c, w, ids),
                lambda a, _, c: mix.moe_output_weighted(x, a, c, w, ids, mix.ACT_CLAMPED, 7.0, 1.7),
                lambda _, b, c: mix.moe_output_weighted(x, b, c, w, ids, mix.ACT_RELU2, 0.0, 0.0),
                lambda a, _, c: ops.moe_apply(x, a, c, w, ids, e)):
        got, want = run(w13, w1, w2).float(), run(off(w13), off(w1), off(w2)).float()
        assert ((got - want).norm() / want.norm()).item() < 2 ** -9   # the library may take another kernel for other strides


def test_many_rows_of_large_experts_take_the_library(cuda, monkeypatch):
    """From GROUPED_MAX_ROWS rows per expert of a large matrix on the library products run (not where a graph is captured, which can't
    read the offsets): the bits of a call whose weights the grouped product does not take (an unaligned start)."""
    from src import ops

    monkeypatch.setattr(mix, "GROUPED_ANY_ROWS_SIZE", 256 * 512)
    monkeypatch.setattr(mix, "GROUPED_MAX_ROWS", 200)
    g = torch.Generator().manual_seed(9)
    h, f, e, k, bf = 256, 512, 3, 2, torch.bfloat16
    w13, w2 = ((torch.randn(*s, generator=g) * 0.05).to(bf).to(cuda) for s in ((e, 2 * f, h), (e, h, f)))
    off = lambda v: torch.empty(v.numel() + 1, dtype=bf, device=cuda)[1:].view(v.shape).copy_(v)
    for t in (299, 300):   # one row short of it, there
        x, w = torch.randn(t, h, generator=g).to(bf).to(cuda), torch.rand(t, k, generator=g).to(cuda)
        ids = torch.rand(t, e, generator=g).argsort(1)[:, :k].int().to(cuda)
        got, want = ops.moe_apply(x, w13, w2, w, ids, e), ops.moe_apply(x, off(w13), off(w2), w, ids, e)
        assert torch.equal(got, want) == (t == 300)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.moe_apply(x, w13, w2, w, ids, e)
    for _ in range(3):
        graph.replay()
        assert ((out - want).float().norm() / want.float().norm()).item() < 1e-2


@pytest.mark.parametrize("tile", [64, 96])   # 64, 128 weight rows
@pytest.mark.parametrize("counts", [(0, 1, 63, 64, 65), (31, 0, 127, 128, 129, 192), (193, 255, 0, 256, 257), (513, 700, 2)])
@pytest.mark.parametrize("K,ncols,act", [(64, 256, mix.MOE_NONE), (256, 128, mix.MOE_SILU), (448, 256, mix.MOE_CLAMPED), (512, 512, mix.MOE_RELU2),
                                         (1088, 384, mix.MOE_GELU), (4096, 256, mix.MOE_NONE)])
def test_small_tiles(cuda, tile, counts, K, ncols, act):
    """Tiles of 64 and 128 weight rows: heights around 64-row pieces, fewer and more stages than LDS holds of each."""
    topk = 2 if sum(counts) % 2 == 0 else 1
    x, w, offsets, idx, scale = _case(counts, K, ncols, act in (mix.MOE_SILU, mix.MOE_CLAMPED, mix.MOE_GELU), topk)
    for rows, sc in ((idx, None), (idx, scale), (None, None)):
        if rows is None and topk > 1:
            continue
        out = torch.full((sum(counts), ncols), float("nan"), dtype=torch.bfloat16, device=cuda)
        dev = [t.to(cuda) if t is not None else None for t in (x, w, offsets, rows, sc)]
        assert mix._kern().moe_gemm(out, *dev[:4], topk if rows is not None else 1, dev[4], act, 1.5, 1.7, tile)
        want = _want(x, w, offsets, rows, topk, act, sc, 1.5, 1.7)
        tol = 2.0 ** -8 * (want.abs() + want.square().mean(1, keepdim=True).sqrt())
        assert ((out.cpu().double() - want).abs() <= tol).all()


@pytest.mark.parametrize("tile,K,ncols,act", [(256, 448, 512, mix.MOE_NONE), (128, 64, 256, mix.MOE_SILU), (160, 1088, 256, mix.MOE_CLAMPED), (0, 640, 512, mix.MOE_RELU2)])
def test_tiles_that_start_within_k(cuda, tile, K, ncols, act):
    """Enough weight tiles that each starts at a stage of its own, beside experts of several row tiles, which start at the first."""
    counts = [3, 0, 1, 300] * 16 + [40] * 8
    x, w, offsets, idx, scale = _case(counts, K, ncols, act in (mix.MOE_SILU, mix.MOE_CLAMPED), 2)
    out = torch.full((sum(counts), ncols), float("nan"), dtype=torch.bfloat16, device=cuda)
    dev = [t.to(cuda) for t in (x, w, offsets, idx, scale)]
    assert mix._kern().moe_gemm(out, *dev[:4], 2, dev[4], act, 1.5, 1.7, tile)
    want = _want(x, w, offsets, idx, 2, act, scale, 1.5, 1.7)
    tol = 2.0 ** -8 * (want.abs() + want.square().mean(1, keepdim=True).sqrt())
    assert ((out.cpu().double() - want).abs() <= tol).all()


@pytest.mark.parametrize("experts,rows,tile", [(16, 40, 96), (16, 80, 96), (16, 81, 256), (32, 60, 96), (32, 61, 256)])
def test_tiles_of_few_rows(cuda, experts, rows, tile):
    """What a step of up to four turns of tiles of 64 weight rows (on 256 compute units), and one of more, takes on either side of its line: the bits of those
    tiles and not of the others, whose sums run in another order."""
    counts = [rows - 7, rows + 7] * (experts // 2)
    x, w, offsets, idx, scale = _case(counts, 512, 4096, False, 2)
    dev = [t.to(cuda) for t in (x, w, offsets, idx)]
    out = {}
    for code in (0, 96, 256):
        out[code] = torch.full((sum(counts), 4096), float("nan"), dtype=torch.bfloat16, device=cuda)
        assert mix._kern().moe_gemm(out[code], *dev, 2, None, mix.MOE_NONE, 1.5, 1.7, code)
    assert torch.equal(out[0], out[tile]) and not torch.equal(out[0], out[96 + 256 - tile])
    rel = ((out[96].float() - out[256].float()).norm() / out[256].float().norm()).item()
    assert rel < 2.0 ** -9   # (rounded to another bf16 now and then)
