"""The expert products of decode steps from unsorted (token, slot) pairs (gemm_decode.hip) against float64: row counts around every
activation image (16, 32, 64, 128), experts without rows and with all of them, ids that name no expert, every activation and tile.

Results are rounded to bf16 once (2^-9 of each value); the fp32 sums add 2^-24 of their terms' size per product, which matters
only beside cancelled values: 2^-8 of the value plus 2^-8 of the row's root mean square covers both."""

import pytest
import torch
import torch.nn.functional as F

from src import ops
from src.ops import mix

pytestmark = pytest.mark.gpu


def _act(z, act):
    if act == mix.MOE_RELU2:
        return torch.relu(z) ** 2
    if act == mix.MOE_NONE:
        return z
    g, u = z.chunk(2, -1)
    if act == mix.MOE_SILU:
        return F.silu(g) * u
    if act == mix.MOE_GELU:
        return F.gelu(g, approximate="tanh") * u
    g, u = g.clamp(max=1.5), u.clamp(-1.5, 1.5)
    return g * torch.sigmoid(1.7 * g) * (u + 1)


def _close(got, want):
    tol = 2.0 ** -8 * (want.abs() + want.square().mean(1, keepdim=True).sqrt())
    return ((got.cpu().double() - want).abs() <= tol).all()


@pytest.mark.parametrize("wr,kc", [(32, 128), (64, 128), (128, 128), (32, 256), (64, 256), (64, 64), (128, 64), (64, 32), (128, 32)])
@pytest.mark.parametrize("act", [mix.MOE_NONE, mix.MOE_SILU, mix.MOE_CLAMPED, mix.MOE_GELU, mix.MOE_RELU2])
def test_products(cuda, wr, kc, act):
    E, N, K, k = 5, 128, 512, 2
    gate = mix.MOE_SILU <= act <= mix.MOE_GELU
    g = torch.Generator().manual_seed(wr + kc + act)
    w = (torch.randn(E, N * (2 if gate else 1), K, generator=g) * K ** -0.5).to(torch.bfloat16)
    ran = 0
    for t in (1, 16, 17, 33, 64, 65, 128):
        x = torch.randn(t, K, generator=g).to(torch.bfloat16)
        ids = torch.rand(t, E + 2, generator=g).argsort(1)[:, :k].int()
        ids[:, 0] = 1                                                    # one expert has every token
        ids[:, 1] = torch.where(ids[:, 1] == 1, E + 1, ids[:, 1])        # E, E + 1: no experts
        y = torch.full((t * k, N), 7.0, dtype=torch.bfloat16, device=cuda)
        if not ops._kern().gemm_decode_ids(y, x.to(cuda), w.to(cuda), ids.reshape(-1).to(cuda), k, t, act, 1.5, 1.7, wr, kc):
            assert not ops.gd_tile_valid(wr, kc, 32 if t <= 32 else 64 if t <= 64 else 128)
            assert (y == 7.0).all()
            continue
        ran += 1
        flat = ids.reshape(-1).long()
        real = flat < E
        want = _act(torch.einsum("nk,nok->no", x.double().repeat_interleave(k, 0)[real], w.double()[flat[real]]), act)
        assert _close(y[real.to(cuda)], want)
        assert (y[~real.to(cuda)] == 7.0).all()
    assert ran


@pytest.mark.parametrize("t", [1, 3, 32, 50, 128])
@pytest.mark.parametrize("H,ff,E,k,n_route", [(512, 256, 4, 2, 6), (256, 192, 40, 4, 40), (320, 96, 6, 1, 6)])
def test_mixtures(cuda, t, H, ff, E, k, n_route):
    """The three mixtures whose decode steps take them, and widths that only narrower tiles (or the sorted products) divide."""
    g = torch.Generator().manual_seed(t + H)
    bf = torch.bfloat16
    x = torch.randn(t, H, generator=g).to(bf)
    w13, w1, w2 = ((torch.randn(*s, generator=g) * s[-1] ** -0.5).to(bf) for s in ((E, 2 * ff, H), (E, ff, H), (E, H, ff)))
    ids = torch.rand(t, n_route, generator=g).argsort(1)[:, :k].int()
    w = torch.rand(t, k, generator=g) + 0.1
    dev = lambda *a: [v.to(cuda) for v in a]
    got = mix.moe_output_weighted(*dev(x, w13, w2, w, ids), mix.ACT_CLAMPED, 1.5, 1.7, n_route=n_route)
    want = mix.ref.moe_output_weighted(x.double(), w13.double(), w2.double(), w.double(), ids, mix.ACT_CLAMPED, 1.5, 1.7, None, None).double()
    assert ((got.cpu().double() - want).norm() / want.norm()).item() < 2 ** -7
    got = mix.moe_output_weighted(*dev(x, w1, w2, w, ids), mix.ACT_RELU2, 0.0, 0.0, n_route=n_route)
    want = mix.ref.moe_output_weighted(x.double(), w1.double(), w2.double(), w.double(), ids, mix.ACT_RELU2, 0.0, 0.0, None, None).double()
    assert ((got.cpu().double() - want).norm() / want.norm()).item() < 2 ** -7
    real = (ids % E).int()
    want = torch.zeros(t, H, dtype=torch.float64)
    plain = torch.zeros(t, H, dtype=torch.float64)
    for j in range(k):
        e = real[:, j].long()
        f = lambda z: torch.einsum("tf,thf->th", _act(torch.einsum("th,tfh->tf", z, w13.double()[e]), mix.MOE_SILU), w2.double()[e])
        want += f((x.double() * w[:, j:j + 1].double()))
        plain += w[:, j:j + 1].double() * f(x.double())
    got = mix.moe_input_scaled(*dev(x, w13, w2, w, real))
    assert ((got.cpu().double() - want).norm() / want.norm()).item() < 2 ** -7
    got = ops.moe_apply(*dev(x, w13, w2, w, real), E)
    assert ((got.cpu().double() - plain).norm() / plain.norm()).item() < 2 ** -7


@pytest.mark.parametrize("t", [3, 40, 100])
@pytest.mark.parametrize("H,ff", [(512, 256), (320, 96)])
def test_rows_and_results_are_formed_once(cuda, monkeypatch, t, H, ff):
    """Whether or not the widths tile, the rows are gathered once and one buffer takes the experts' results."""
    E, k, bf = 4, 2, torch.bfloat16
    x, w13, w2 = (torch.randn(*s, device=cuda).to(bf) for s in ((t, H), (E, 2 * ff, H), (E, H, ff)))
    w, ids = torch.rand(t, k, device=cuda), torch.randint(0, E, (t, k), device=cuda, dtype=torch.int32)

    class Counting:
        gathers = 0

        def __init__(self, kern):
            self.kern = kern

        def __getattr__(self, name):
            Counting.gathers += name == "gather_scaled"
            return getattr(self.kern, name)

    kern = Counting(mix._kern())
    monkeypatch.setattr(mix, "_kern", lambda: kern)
    mix.moe_input_scaled(x, w13, w2, w, ids)
    assert Counting.gathers == 1
    made = []
    zeros = torch.zeros
    monkeypatch.setattr(torch, "zeros", lambda *a, **kw: (made.append(a), zeros(*a, **kw))[1])
    ops.moe_apply(x, w13, w2, w, ids, E + 1)
    assert made.count((t * k, H)) == 1


@pytest.mark.parametrize("H,ff,t,form", [(4096, 2048, 1, "ids"), (4096, 2048, 2, "grouped"), (4096, 2048, 32, "grouped"), (4096, 2048, 33, "ids"),
                                         (6144, 2048, 8, "grouped"), (4096, 1024, 8, "ids"), (2048, 2048, 32, "ids"), (5120, 2048, 8, "ids"), (4096, 4096, 2, "ids"), (4096, 4096, 32, "ids")])
def test_scaled_mixtures_whose_sorted_form_is_faster_keep_it(cuda, monkeypatch, H, ff, t, form):
    """Large gated experts with weight rows of a multiple of 4 KiB and fewer than 4096 columns, 2 to 32 tokens: sorted rows, tiles of 32 weight rows."""
    E, k, bf, ran = 3, 2, torch.bfloat16, []
    g = torch.Generator(device=cuda).manual_seed(H + t)
    x, w13, w2 = (torch.randn(*s, generator=g, device=cuda).to(bf) for s in ((t, H), (E, 2 * ff, H), (E, H, ff)))
    w13, w2 = w13 * 2.0 ** -6, w2 * 2.0 ** -6
    w, ids = torch.rand(t, k, generator=g, device=cuda) + 0.1, torch.rand(t, E, generator=g, device=cuda).argsort(1)[:, :k].int().contiguous()

    class Recording:
        def __init__(self, kern):
            self.kern = kern

        def __getattr__(self, name):
            ran.append(name)
            return getattr(self.kern, name)

    kern = Recording(ops._kern())
    monkeypatch.setattr(ops, "_kern", lambda: kern)
    got = mix.moe_input_scaled(x, w13, w2, w, ids)
    assert ran == [f"gemm_decode_{form}"] * 2
    want = torch.zeros(t, H, dtype=torch.float64, device=cuda)
    for e in range(E):
        for j in range(k):
            rows = (ids[:, j] == e).nonzero().flatten()
            want[rows] += _act((x[rows].double() * w[rows, j:j + 1].double()) @ w13[e].double().T, mix.MOE_SILU) @ w2[e].double().T
    assert ((got.double() - want).norm() / want.norm()).item() < 2 ** -7
