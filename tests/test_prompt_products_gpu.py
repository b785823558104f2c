"""The dense products of prompt steps (moe_gemm.hip with parts of K, or with the gate), their consumers and the rules that choose them.

Slabs are fp32 sums of K / sk products of bf16 values: terms of size s give an error of about sqrt(K) 2^-24 s sqrt(K) at the worst, 2^-24 K of the
row's root mean square; 2^-20 sqrt(K) of it covers the order of the sums and is far below what a wrong row, column or stage moves. bf16 results
are rounded once: 2^-8 of the value plus 2^-8 of the rows' root mean square."""

import pytest
import torch
import torch.nn.functional as F

from src import ops


def _xw(m, n, k, seed=0):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(m, k, generator=g).bfloat16(), (torch.randn(n, k, generator=g) * k ** -0.5).bfloat16()


def _close(got, want, rel):
    got, want = got.double().cpu(), want.double()
    assert bool(((got - want).abs() <= rel * want.abs() + rel * want.square().mean().sqrt()).all())


# rows: one, around tiles of 64 and 256 and their even shares, several row tiles; parts of one stage and of several; every tile code
@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 63, 129, 192, 255, 256, 257, 300, 513, 769])
@pytest.mark.parametrize("n,k,sk,code", [(256, 64, 1, 0), (256, 512, 8, 96), (512, 192, 3, 64), (768, 1024, 4, 0), (1024, 448, 7, 96), (256, 2048, 2, 224)])
def test_slabs(m, n, k, sk, code):
    x, w = _xw(m, n, k)
    slab = torch.full((sk, m, n), float("nan"), device="cuda")
    ops._kern().dense_gemm(slab, x.cuda(), w.cuda(), None, code)
    want = x.double() @ w.double().t()
    _close(slab.double().sum(0), want, 2.0 ** -20 * k ** 0.5)
    part = k // sk
    for e in (0, sk - 1):   # every slab is its part of K
        at = slice(e * part, (e + 1) * part)
        _close(slab[e], x[:, at].double() @ w[:, at].double().t(), 2.0 ** -20 * k ** 0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 129, 168, 256, 257, 511, 800])
@pytest.mark.parametrize("inter,k,code", [(128, 64, 0), (384, 512, 96), (256, 192, 64), (640, 1024, 0)])
def test_gate_on_sums(m, inter, k, code):
    x, w = _xw(m, 2 * inter, k)
    scale = torch.rand(m, generator=torch.Generator().manual_seed(1)) + 0.5
    z = (x.double() @ w.double().t()) * scale.double()[:, None]
    want = F.silu(z[:, :inter]) * z[:, inter:]
    wide = torch.zeros(m, k + 8, dtype=torch.bfloat16, device="cuda")
    wide[:, :k] = x.cuda()
    for rows in (x.cuda(), wide[:, :k]):   # rows K and more apart
        out = torch.empty(m, inter, dtype=torch.bfloat16, device="cuda")
        ops._kern().dense_gemm(out, rows, w.cuda(), scale.cuda(), code)
        _close(out, want, 2.0 ** -8)


@pytest.mark.gpu
@pytest.mark.parametrize("t,h,sk", [(129, 4096, 8), (300, 8192, 1), (1, 1024, 3), (513, 2056, 5)])
def test_row_scale_after_slabs(t, h, sk):
    g = torch.Generator().manual_seed(0)
    res = torch.randn(t, h, generator=g).bfloat16().cuda()
    slab = torch.randn(sk, t, h, generator=g).cuda()
    want = res.double() + slab.double().sum(0)
    rs = ops.rms_row_scale_slab(res, slab, 1e-5)
    _close(res, want.cpu(), 2.0 ** -8)
    # the statistics are those of the rounded rows
    assert torch.allclose(rs.double(), torch.rsqrt(res.double().square().mean(-1) + 1e-5), rtol=1e-5, atol=0)


@pytest.mark.gpu
def test_rope_of_scaled_slabs():
    t, hq, hkv, d, nb = 131, 4, 2, 128, 9
    g = torch.Generator().manual_seed(0)
    slab, rs = torch.randn(4, t, (hq + 2 * hkv) * d, generator=g).cuda(), (torch.rand(t, generator=g) + 0.5).cuda()
    cs = torch.randn(200, d, generator=g).cuda()
    pos = torch.arange(t, device="cuda")

    def rows(s, scale):
        k, v = (torch.zeros(nb, hkv, 16, d, dtype=torch.bfloat16, device="cuda") for _ in range(2))
        return ops.rope_and_cache_slab(s, pos, cs, pos, k, v, hq, hkv, d, row_scale=scale), k, v

    for a, b in zip(rows(slab, rs), rows(slab.sum(0, keepdim=True) * rs[None, :, None], None)):
        _close(a, b.double().cpu(), 2.0 ** -8)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [129, 200, 257, 600])
@pytest.mark.parametrize("keep", [False, True])
def test_steps_of_few_row_tiles(monkeypatch, rows, keep):
    """A prompt step with every product by slabs and the gate on sums against the library's products: one bf16 rounding apart per product."""
    from src.models.llama import AttnMetadata, CausalLM
    from src.models.presets import get_preset

    m = CausalLM(get_preset("llama-mini"), "cuda:0", seed=3, max_position=1024, full_init=True)
    nb = (rows + 15) // 16
    ids = torch.randint(3, 32000, (rows,), generator=torch.Generator().manual_seed(1)).cuda()
    pos = torch.arange(rows, device="cuda")
    cu = torch.tensor([0, rows - 100, rows], dtype=torch.int32, device="cuda")
    pos = torch.cat([pos[: rows - 100], pos[:100]])
    tables = torch.arange(2 * nb, dtype=torch.int32, device="cuda").view(2, nb)
    slots = torch.cat([pos[: rows - 100], nb * 16 + pos[rows - 100:]])
    got = []
    for own in (True, False):
        if own:   # (the rules leave products of these widths to the library)
            monkeypatch.setattr(ops, "prompt_slab_parts", lambda mm, n, k, cus, residual: ops.slab_parts(mm, n, k, cus))
            monkeypatch.setattr(ops, "prompt_silu_tiles", lambda mm, *a: 96 if mm <= 256 else 0)
        else:
            monkeypatch.setattr(ops, "_dense_gemm_ok", lambda x, w: False)
        pool = torch.zeros(m.arch.num_layers, 2, 2 * nb, m.hkv, 16, 128, dtype=m.dtype, device="cuda")
        meta = AttnMetadata(True, slots, tables, torch.tensor([rows - 100, 100], dtype=torch.int32, device="cuda"), cu, max(rows - 100, 100),
                            keep_rows=(cu[1:] - 1).long() if keep else None)
        got.append((m.forward(ids, pos, meta, pool).double(), pool.double()))
    for a, b in zip(*got):
        assert float((a - b).norm() / b.norm()) < 2e-2


def test_parts_of_k():
    """Parts are whole stages of K, one workgroup per compute unit at most."""
    for m in (129, 224, 256, 257, 512, 1000, 2048, 5000):
        for n, k in ((4096, 4096), (4096, 14336), (6144, 4096), (8192, 28672), (1024, 2048), (256, 64), (768, 192)):
            sk, code = ops.slab_parts(m, n, k, 256)
            assert 1 <= sk <= 8 and k % (64 * sk) == 0 and (sk == 1 or (n // 128 if code == 96 else n // 256 * -(-m // 256)) * sk <= 256)
    x, w = torch.zeros(300, 64, dtype=torch.bfloat16), torch.zeros(256, 64, dtype=torch.bfloat16)
    assert ops.prompt_slab(x, w) is None   # (not on a device)


@pytest.mark.parametrize("n,k,residual,own,library", [
    # qkv: either side of the lines in rows, columns and K; small models and shards
    (6144, 4096, False, {129: 4, 256: 4}, [257, 300]), (5120, 8192, False, {160: 4, 256: 4}, [129, 159, 257]), (4608, 3072, False, {160: 6, 256: 6}, [129, 300]),
    (6144, 2560, False, {129: 5, 256: 5}, [300]), (6144, 2048, False, {}, [129, 160, 256]), (3840, 5120, False, {}, [129, 256]), (3072, 4096, False, {}, [129, 256]),
    (1536, 1024, False, {}, [129, 256]), (1536, 4096, False, {}, [129, 256]), (1280, 8192, False, {}, [129, 256]), (10240, 8192, False, {}, [129, 256]),
    # o and down
    (4096, 14336, True, {129: 8, 256: 8, 257: 8, 1024: 4, 2048: 2}, [2300]), (4096, 11008, True, {192: 4, 257: 4, 768: 4}, [193, 256, 769]),
    (2560, 9728, True, {129: 8, 256: 8, 768: 8}, [769]), (2048, 5632, True, {129: 8, 192: 8}, [193, 256, 257]), (5120, 5120, True, {129: 5, 224: 5}, [225, 300]),
    (4096, 4096, True, {129: 8, 192: 8}, [193, 224, 300]), (3072, 3072, True, {129: 8, 192: 8}, [193, 256]), (2560, 4096, True, {}, [129, 192, 224, 300]),
    (2048, 2048, True, {}, [129, 192, 224]), (1024, 1024, True, {}, [129, 224])])
def test_choice_of_slabs(n, k, residual, own, library):
    """The parts that are taken, and where the library is, on a device of 256 compute units."""
    for m, sk in own.items():
        assert ops.prompt_slab_parts(m, n, k, 256, residual) == (sk, 96 if m <= 256 else 0)
    assert all(ops.prompt_slab_parts(m, n, k, 256, residual) is None for m in library)


@pytest.mark.parametrize("inter,k,own,library", [
    (14336, 4096, {129: 96, 256: 96, 257: 0, 600: 0, 3072: 0}, [3073]), (11008, 4096, {129: 96, 192: 96, 257: 0, 769: 0}, [193, 256, 513, 768]),
    (9728, 2560, {129: 96, 192: 96, 257: 0}, [193, 256]), (8192, 2048, {513: 0, 2500: 0}, [129, 256, 257, 512]), (13824, 5120, {257: 0, 1000: 0}, [129, 160, 256, 1537]),
    (28672, 8192, {129: 0, 168: 0, 257: 0, 1536: 0}, [169, 256, 1537]), (4096, 2048, {1281: 0, 2500: 0}, [129, 256, 300, 1000, 1024]), (2048, 1024, {}, [129, 160, 256, 300, 1500, 2500])])
def test_choice_of_gate_tiles(inter, k, own, library):
    """Tiles of the gate and up product, and where the library's is taken, on a device of 256 compute units."""
    assert {m: ops.prompt_silu_tiles(m, inter, k, 256) for m in own} == own
    assert all(ops.prompt_silu_tiles(m, inter, k, 256) is None for m in library)
