"""Attention of prompt-sized steps: the 16-rows-per-wave matrix-core kernel against the fp32 FMA kernel, at remainders of its row and
key tiles, in every score form, and over more keys than its row table holds. Weights are rounded to bf16 on the matrix-core side
(2^-9 of sum w |v|), results on both (2^-8 each). The same inputs with the keys split go through the other kernel and the merge."""

import pytest
import torch

from src.ops import seq

pytestmark = pytest.mark.gpu


def _forms(monkeypatch):
    """The forms that sink_attn's launches took, in a list that grows with every call."""
    kern, forms = seq._kern(), []

    class Spy:
        def __getattr__(self, name):
            if name != "sink_attn":
                return getattr(kern, name)
            return lambda *a: forms.append(kern.sink_attn(*a))

    monkeypatch.setattr(seq, "_kern", lambda: Spy())
    return forms


def _kernels(monkeypatch):
    """The same with the kernels of the forms that have several."""
    kern, names = seq._kern(), []

    class Spy:
        def __getattr__(self, name):
            if name != "sink_attn":
                return getattr(kern, name)
            return lambda *a: names.append(kern.sink_attn_named(*a))

    monkeypatch.setattr(seq, "_kern", lambda: Spy())
    return names


@pytest.mark.parametrize("seqs", [2, 72])   # 2: the keys are split, and the 32-rows-per-wave kernel runs; 72: enough row tiles without
@pytest.mark.parametrize("dim,vdim,heads,groups,bs,style,past", [
    (128, 128, 16, 4, 16, "", 0), (64, 64, 15, 5, 32, "sink", 70), (64, 128, 16, 4, 16, "cap", 5), (64, 256, 16, 4, 16, "bias", 33), (128, 128, 16, 4, 16, "bias", 0),
    (128, 64, 16, 4, 8, "sigmoid", 60), (128, 256, 16, 4, 16, "window", 100), (128, 128, 12, 4, 1, "seg", 0), (128, 128, 16, 4, 4, "", 1300),
    (128, 128, 16, 4, 16, "slopes", 200), (64, 64, 16, 4, 16, "sigmoid", 0)])
def test_against_fma(cuda, monkeypatch, dim, vdim, heads, groups, bs, style, past, seqs):
    forms = _forms(monkeypatch)
    torch.manual_seed(dim + vdim + heads)
    lens = ([130, 1, 33, 2, 63, 31, 127, 48] * 9)[:seqs]
    pasts = [past + 7 * (s % 3) if past else 0 for s in range(seqs)]
    T, need = sum(lens), [-(-(n + p) // bs) for n, p in zip(lens, pasts)]
    pool = 1 + max(need) * 3
    cache = torch.randn(pool, bs, groups * (dim + vdim), device=cuda).to(torch.bfloat16)
    bt = torch.randint(0, pool, (seqs, max(need)), device=cuda, dtype=torch.int32)
    cu = torch.tensor([0] + lens, device=cuda).cumsum(0).int()
    pos = torch.cat([torch.arange(n) + p for n, p in zip(lens, pasts)]).to(cuda)
    ctx = torch.tensor([n + p for n, p in zip(lens, pasts)], device=cuda, dtype=torch.int32)
    q = torch.randn(T, heads * dim, device=cuda).to(torch.bfloat16)
    f = lambda *s: torch.randn(*s, device=cuda)
    sink, bias, window, kw = None, None, 0, {}
    if style == "sink":
        sink = f(heads) + 2
    if style == "bias":
        sink, bias = f(heads), f(40, heads)
    if style == "cap":
        kw = dict(softcap=5.0, slopes=torch.rand(heads, device=cuda) * 0.1)
    if style == "slopes":
        kw = dict(slopes=torch.rand(heads, device=cuda) * 0.1)
    if style == "sigmoid":
        kw = dict(sigmoid=True, head_bias=f(heads) - 3)
    if style == "seg":
        kw = dict(seg=100)
    if style == "window":
        window = 70
    args = (q, cache, bt, cu, ctx, pos, sink, bias, max(lens), heads, groups, dim, vdim, window, dim ** -0.5)
    want, got = seq.sink_attn(*args, impl=1, **kw).float(), seq.sink_attn(*args, impl=2, **kw).float()
    mass = 1.0 if style != "sigmoid" else max(lens) + past + 14   # sigmoid weights do not sum to one
    assert forms == ["fma", "rows" if seqs == 72 else "split"]
    top = mass * float(cache.float().abs().max())
    assert ((got - want).abs() <= 2 ** -8.5 * top + 2 ** -7 * want.abs()).all()
    # the bound above is for one key that has it all; over a row the roundings average out
    assert ((got - want).norm() / want.norm()).item() < 2 ** -7


@pytest.mark.parametrize("dim,vdim", [(128, 128), (64, 64), (64, 256)])
@pytest.mark.parametrize("rows,style", [(1, ""), (2, "slopes"), (20, ""), (33, "cap"), (64, ""), (400, "")])
def test_distance_bias_where_distances_end(cuda, monkeypatch, dim, vdim, rows, style):
    """A bias per distance whose table ends within a lane's keys, at their first and last, and beyond all of them: keys so far back
    that all share its last row are not looked up. Unsplit keys, the 16-rows-per-wave kernel."""
    torch.manual_seed(rows + dim)
    forms, heads, groups, bs, seqs = _forms(monkeypatch), 16, 4, 16, 72
    lens = ([130, 1, 33, 2, 63, 31, 127, 48] * 9)[:seqs]
    pasts, T, need = [11 * (s % 4) for s in range(seqs)], sum(lens), 12
    cache = torch.randn(40, bs, groups * (dim + vdim), device=cuda).to(torch.bfloat16)
    bt = torch.randint(0, 40, (seqs, need), device=cuda, dtype=torch.int32)
    cu = torch.tensor([0] + lens, device=cuda).cumsum(0).int()
    pos = torch.cat([torch.arange(n) + p for n, p in zip(lens, pasts)]).to(cuda)
    ctx = torch.tensor([n + p for n, p in zip(lens, pasts)], device=cuda, dtype=torch.int32)
    q = torch.randn(T, heads * dim, device=cuda).to(torch.bfloat16)
    bias = torch.randn(rows, heads, device=cuda) * 2
    kw = {"cap": dict(softcap=5.0), "slopes": dict(slopes=torch.rand(heads, device=cuda) * 0.1)}.get(style, {})
    args = (q, cache, bt, cu, ctx, pos, None, bias, max(lens), heads, groups, dim, vdim, 0, dim ** -0.5)
    want, got = seq.sink_attn(*args, impl=1, **kw).float(), seq.sink_attn(*args, impl=2, **kw).float()
    assert forms == ["fma", "rows"]
    assert ((got - want).abs() <= 2 ** -8.5 * float(cache.float().abs().max()) + 2 ** -7 * want.abs()).all()
    assert ((got - want).norm() / want.norm()).item() < 2 ** -7


def _ragged(cuda, lens, pasts, bs, groups, dim, vdim, heads):
    T, need = sum(lens), max(-(-(n + p) // bs) for n, p in zip(lens, pasts))
    cache = torch.randn(1 + 3 * need, bs, groups * (dim + vdim), device=cuda).to(torch.bfloat16)
    bt = torch.randint(0, 1 + 3 * need, (len(lens), need), device=cuda, dtype=torch.int32)
    cu = torch.tensor([0] + lens, device=cuda).cumsum(0).int()
    pos = torch.cat([torch.arange(n) + p for n, p in zip(lens, pasts)]).to(cuda)
    ctx = torch.tensor([n + p for n, p in zip(lens, pasts)], device=cuda, dtype=torch.int32)
    return torch.randn(T, heads * dim, device=cuda).to(torch.bfloat16), cache, bt, cu, ctx, pos


@pytest.mark.parametrize("dim,vdim,heads,groups,bs,style", [
    (128, 128, 16, 4, 16, ""), (64, 64, 20, 5, 4, "sink"), (64, 128, 16, 4, 16, "window"), (128, 64, 16, 4, 8, "sigmoid"), (64, 256, 12, 4, 16, ""),
    (128, 256, 16, 4, 1, "sink"), (128, 128, 12, 4, 16, "seg")])
def test_many_rows_of_long_keys(cuda, monkeypatch, dim, vdim, heads, groups, bs, style):
    """128 rows per workgroup: four of them per compute unit, tiles of 64 keys (vdim 256: 32), row counts around 32 and 128, pairs of
    sequence and head that are and are not a multiple of 8."""
    torch.manual_seed(dim + vdim + heads)
    forms = _kernels(monkeypatch)
    lens = ([200, 8, 33, 1, 65, 32, 129, 190] * 11)[:88 if style else 81]
    data = _ragged(cuda, lens, [520 + 7 * (s % 9) for s in range(len(lens))], bs, groups, dim, vdim, heads)
    sink, kw = (torch.randn(heads, device=cuda) if style == "sink" else None), {}
    if style == "sigmoid":
        kw = dict(sigmoid=True, head_bias=torch.randn(heads, device=cuda) - 5)
    if style == "seg":
        kw = dict(seg=512)
    args = (*data, sink, None, max(lens), heads, groups, dim, vdim, 400 if style == "window" else 0, dim ** -0.5)
    want, got = seq.sink_attn(*args, impl=1, **kw).float(), seq.sink_attn(*args, **kw).float()
    assert forms == ["fma", "wide"]
    mass = 1.0 if style != "sigmoid" else 20.0   # of the sigmoid weights
    assert ((got - want).abs() <= 2 ** -8.5 * mass * float(data[1].float().abs().max()) + 2 ** -7 * want.abs()).all()
    assert ((got - want).norm() / want.norm()).item() < 2 ** -7


@pytest.mark.parametrize("seqs,rows,past,form", [(2, 300, 0, "rows"), (8, 128, 0, "rows"), (1, 64, 30, "rows"), (1, 20, 5000, "split"), (3, 9, 1000, "split"),
                                                 (2, 22, 304, "split"), (1, 20, 300, "split")])
def test_keys_are_split_behind_few_rows_only(cuda, monkeypatch, seqs, rows, past, form):
    torch.manual_seed(rows)
    forms = _forms(monkeypatch)
    data = _ragged(cuda, [rows - s for s in range(seqs)], [past] * seqs, 16, 4, 128, 128, 16)
    args = (*data, None, None, rows, 16, 4, 128, 128, 0, 128 ** -0.5)
    want, got = seq.sink_attn(*args, impl=1).float(), seq.sink_attn(*args).float()
    assert forms == ["fma", form]
    assert ((got - want).norm() / want.norm()).item() < 2 ** -7


@pytest.mark.parametrize("rows,past,cap,vdim,form", [(700, 900, 0.0, 128, "rows"), (700, 900, 30.0, 256, "rows"), (40, 4000, 30.0, 128, "split")])
def test_a_window_bounds_the_keys_that_splits_are_weighed_by(cuda, monkeypatch, rows, past, cap, vdim, form):
    torch.manual_seed(rows)
    forms = _forms(monkeypatch)
    data = _ragged(cuda, [rows], [past], 16, 4, 128, vdim, 16)
    args, kw = (*data, None, None, rows, 16, 4, 128, vdim, 500 if rows > 64 else 2000, 128 ** -0.5), {"softcap": cap} if cap else {}
    want, got = seq.sink_attn(*args, impl=1, **kw).float(), seq.sink_attn(*args, **kw).float()
    assert forms == ["fma", form]
    assert ((got - want).norm() / want.norm()).item() < 2 ** -7


@pytest.mark.parametrize("dim,vdim", [(64, 64), (64, 256), (128, 128)])
@pytest.mark.parametrize("style", ["", "sink", "sigmoid", "capped"])
def test_infinite_values_stay_infinite(cuda, monkeypatch, dim, vdim, style):
    """A value of either infinity at a key that every row sees, where weights go in two parts: the same infinity, and the other columns as
    they are without it."""
    torch.manual_seed(dim + vdim)
    forms, heads, groups, bs = _forms(monkeypatch), 16, 4, 16
    q, cache, bt, cu, ctx, pos = _ragged(cuda, [150, 77, 99], [0, 30, 8], bs, groups, dim, vdim, heads)
    bt = torch.arange(bt.numel(), device=cuda, dtype=torch.int32).view_as(bt)
    cache = torch.randn(bt.numel(), bs, groups * (dim + vdim), device=cuda).to(torch.bfloat16)
    sink, kw = (torch.randn(heads, device=cuda) if style == "sink" else None), {}
    if style == "sigmoid":
        kw = dict(sigmoid=True, head_bias=torch.randn(heads, device=cuda) - 5)
    if style == "capped":
        kw = dict(softcap=20.0)
    tail = (bt, cu, ctx, pos, sink, None, 150, heads, groups, dim, vdim, 0, dim ** -0.5)
    plain = seq.sink_attn(q, cache, *tail, **kw).view(-1, heads, vdim)
    first = cache.view(-1, groups, bs, dim + vdim)[:, :, 0]   # of every block; of block bt[s, 0] the sequence's token 0
    first[bt[:, 0].long(), :, dim + 3], first[bt[:, 0].long(), :, dim + 40] = float("inf"), float("-inf")
    got = seq.sink_attn(q, cache, *tail, **kw).view(-1, heads, vdim)
    assert forms == ["rows", "rows"]
    assert (got[:, :, 3] == float("inf")).all() and (got[:, :, 40] == float("-inf")).all()
    rest = [c for c in range(vdim) if c not in (3, 40)]
    assert torch.equal(got[:, :, rest], plain[:, :, rest])


@pytest.mark.parametrize("style,vdim", [("", 128), ("sink", 64), ("capped", 128), ("bias", 256), ("sigmoid", 128)])
def test_fewer_splits_are_no_further_from_64_bits(cuda, monkeypatch, style, vdim):
    """Steps whose keys the rule cuts into fewer splits than there could be: their weights go in two bf16 parts (softmax), so that the results
    are no further from float64 than with all splits, which impl 2 takes. (1 % for the roundings of the results themselves.)"""
    torch.manual_seed(vdim)
    heads, groups, dim = 16, 4, 128 if vdim > 64 else 64
    q, cache, bt, cu, ctx, pos = _ragged(cuda, [150, 140, 133], [1500, 1400, 1333], 16, groups, dim, vdim, heads)
    sink, bias = (torch.randn(heads, device=cuda) if style == "sink" else None), (torch.randn(64, heads, device=cuda) if style == "bias" else None)
    kw = dict(softcap=20.0) if style == "capped" else dict(sigmoid=True, head_bias=torch.randn(heads, device=cuda) - 5) if style == "sigmoid" else {}
    call = lambda impl: seq.sink_attn(q, cache, bt, cu, ctx, pos, sink, bias, 150, heads, groups, dim, vdim, 0, dim ** -0.5, impl, **kw)
    forms = _forms(monkeypatch)
    got, all_splits = call(0), call(2)
    assert forms == ["split", "split"]
    cpu = lambda x: x if x is None else x.cpu()
    want = seq.sink_attn(*(cpu(x) for x in (q.float(), cache.float(), bt, cu, ctx, pos, sink, bias)), 150, heads, groups, dim, vdim, 0, dim ** -0.5,
                         **{k: cpu(v) if torch.is_tensor(v) else v for k, v in kw.items()})
    error = lambda x: ((x.cpu().double() - want.double()).norm() / want.double().norm()).item()
    assert error(got) <= 1.01 * error(all_splits)


@pytest.mark.parametrize("kernel,dim,vdim,style,seqs,past", [
    ("wide", 128, 128, "", 76, 1150), ("wide", 64, 256, "sink", 76, 1060), ("wide", 64, 64, "sigmoid", 76, 2200), ("rows", 128, 128, "cap", 72, 1150),
    ("rows", 64, 64, "bias", 72, 2200), ("rows", 64, 256, "slopes", 72, 1100), ("fine rows", 128, 128, "", 50, 1300), ("fine rows", 64, 128, "sigmoid", 50, 1300),
    ("fine rows", 128, 256, "sink", 40, 1100)])
def test_row_table_is_filled_again(cuda, monkeypatch, kernel, dim, vdim, style, seqs, past):
    """More visible keys than the 1024 rows that a workgroup's table of cache rows holds, for every kernel that has one."""
    torch.manual_seed(dim + vdim + seqs)
    names, heads, groups = _kernels(monkeypatch), 16, 4
    data = _ragged(cuda, ([130, 1, 33, 2, 63, 31, 127, 48] * 10)[:seqs], [past + 7 * (s % 3) for s in range(seqs)], 16, groups, dim, vdim, heads)
    f = lambda *s: torch.randn(*s, device=cuda)
    sink, bias, kw = (f(heads) if style == "sink" else None), (f(40, heads) if style == "bias" else None), {}
    if style == "cap":
        kw = dict(softcap=5.0, slopes=torch.rand(heads, device=cuda) * 0.01)
    if style == "slopes":
        kw = dict(slopes=torch.rand(heads, device=cuda) * 0.01)
    if style == "sigmoid":
        kw = dict(sigmoid=True, head_bias=f(heads) - 5)
    args = (*data, sink, bias, 130, heads, groups, dim, vdim, 0, dim ** -0.5)
    want, got = seq.sink_attn(*args, impl=1, **kw).float(), seq.sink_attn(*args, **kw).float()
    assert names == ["fma", kernel]
    mass = 1.0 if style != "sigmoid" else 40.0   # of the sigmoid weights
    assert ((got - want).abs() <= 2 ** -8.5 * mass * float(data[1].float().abs().max()) + 2 ** -7 * want.abs()).all()
    assert ((got - want).norm() / want.norm()).item() < 2 ** -7


@pytest.mark.parametrize("dim,vdim", [(64, 64), (64, 128), (64, 256), (128, 64), (128, 128), (128, 256)])
@pytest.mark.parametrize("style", ["sigmoid", "sink", "bias", "cap", "window"])
def test_weights_in_two_parts(cuda, monkeypatch, dim, vdim, style):
    """Every width and kind of scores of the steps whose weights go in two bf16 parts. The weights' own rounding is gone (2^-17 of sum w |v|
    is left), so results are within their one rounding, 2^-9, of the fp32 kernel's before its rounding: 2^-8 of both, and 2^-12 for sums of cancelled values."""
    torch.manual_seed(dim + vdim)
    names, heads, groups = _kernels(monkeypatch), 16, 4
    data = _ragged(cuda, [150, 1, 77, 33], [0, 40, 21, 64], 16, groups, dim, vdim, heads)
    f = lambda *s: torch.randn(*s, device=cuda)
    sink, bias, window, kw = (f(heads) if style == "sink" else None), (f(40, heads) if style == "bias" else None), 50 if style == "window" else 0, {}
    if style == "cap":
        kw = dict(softcap=5.0, slopes=torch.rand(heads, device=cuda) * 0.1)
    if style == "sigmoid":
        kw = dict(sigmoid=True, head_bias=f(heads) - 3)
    args = (*data, sink, bias, 150, heads, groups, dim, vdim, window, dim ** -0.5)
    want, got = seq.sink_attn(*args, impl=1, **kw).float(), seq.sink_attn(*args, **kw).float()
    assert names == ["fma", "fine rows"]
    mass = 1.0 if style != "sigmoid" else 150.0   # of the sigmoid weights
    assert ((got - want).abs() <= 2 ** -12 * mass * float(data[1].float().abs().max()) + 2 ** -7 * want.abs()).all()
    assert ((got - want).norm() / want.norm()).item() < 2 ** -8
