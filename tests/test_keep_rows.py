"""The rows that a prompt step's last layer goes on with, in one launch against the same gathers (copies: equal to the bit)."""

import pytest
import torch

from src import ops


def _step(dev, lens, width=24, hidden=40, extra=16, blocks=5):
    g = torch.Generator().manual_seed(0)
    t, s = sum(lens), len(lens)
    cu = torch.tensor([0] + lens).cumsum(0).int()
    wide = torch.randn(t, width + extra, generator=g).bfloat16()
    tables = torch.randint(0, 99, (s, blocks + 3), generator=g, dtype=torch.int32)
    args = [cu, tables, torch.randint(1, 99, (s,), generator=g, dtype=torch.int32), wide, torch.randn(t, hidden, generator=g).bfloat16(), torch.rand(t, generator=g)]
    cu, tables, ctx, wide, resid, rs = (a.to(dev) for a in args)
    return cu, tables[:, :blocks], ctx, wide, width, resid, rs


def _want(keep, cu, tables, ctx, q, width, resid, rs):
    seq = [next(i for i in range(len(cu) - 1) if int(cu[i + 1]) > int(k)) for k in keep]
    return q[keep, :width], resid[keep], tables[seq], ctx[seq], torch.arange(len(keep) + 1, dtype=torch.int32), rs[keep] if rs is not None else None


# one sequence, empty ones between, more sequences than a workgroup has threads; first, inner and last rows; with and without scales
@pytest.mark.parametrize("lens", [[7], [1, 0, 0, 5, 3, 0], [2] * 600])
@pytest.mark.parametrize("scaled", [True, False])
@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_rows(dev, lens, scaled):
    cu, tables, ctx, q, width, resid, rs = _step(dev, lens)
    rs = rs if scaled else None
    ends = [int(e) - 1 for e, n in zip(cu[1:], lens) if n > 0]
    for keep in (ends, [0], list(range(sum(lens)))[::3][::-1]):
        at = torch.tensor(keep, dtype=torch.int64)
        got = ops.keep_rows(at.to(dev), cu, tables, ctx, q, width, resid, rs)
        want = _want(at, cu.cpu(), tables.cpu(), ctx.cpu(), q.cpu(), width, resid.cpu(), rs.cpu() if scaled else None)
        for a, b in zip(got, want):
            assert (a is None) == (b is None)
            if a is not None:
                assert a.dtype == b.dtype and a.is_contiguous() and torch.equal(a.cpu(), b)


@pytest.mark.gpu
@pytest.mark.parametrize("scaled", [True, False])
def test_turned_queries(scaled):
    """Heads of 128 turned at their sequence's last position and scaled, against the plain form in torch: the same fp32 terms, rounded to bf16 once
    (2^-8 of the pair covers a sum next to a tie)."""
    cu, tables, ctx, q, width, resid, rs = _step("cuda", [3, 1, 0, 9], width=384)
    cs = torch.randn(60, 128, generator=torch.Generator().manual_seed(1)).cuda()   # (fewer positions than the longest context: the last one)
    keep = torch.tensor([2, 3, 12], device="cuda")
    got = ops.keep_rows(keep, cu, tables, ctx, q, width, resid, rs if scaled else None, cos_sin=cs)
    want = ops.keep_rows(keep.cpu(), cu.cpu(), tables.cpu(), ctx.cpu(), q.cpu(), width, resid.cpu(), rs.cpu() if scaled else None, cos_sin=cs.cpu())
    assert got[5] is None and want[5] is None and all(torch.equal(a.cpu(), b) for a, b in zip(got[1:5], want[1:5]))
    a, b = got[0].float().cpu().view(3, 3, 2, 64), want[0].float().view(3, 3, 2, 64)
    assert bool(((a - b).abs() <= 2.0 ** -8 * b.norm(dim=2, keepdim=True)).all())


@pytest.mark.parametrize("scaled", [True, False])
@pytest.mark.parametrize("turned", [True, False])
@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_rows_outside_the_step(dev, scaled, turned):
    """Refused on the CPU; NaN on the GPU, never another row's values, beside rows that are as ever."""
    cu, tables, ctx, q, width, resid, rs = _step(dev, [3, 1, 0, 9], width=384)
    args = (cu, tables, ctx, q, width, resid, rs if scaled else None, torch.ones(60, 128, device=dev) if turned else None)
    keep = torch.tensor([-1, 13, 12, 2 ** 40], device=dev)
    if dev == "cpu":
        for at in (keep[:1], keep[1:2], keep[3:]):
            with pytest.raises((IndexError, RuntimeError)):
                ops.keep_rows(at, *args)
        return
    got, inner = ops.keep_rows(keep, *args), ops.keep_rows(keep[2:3], *args)
    for a, b in zip(got[:2] + got[5:], inner[:2] + inner[5:]):
        if a is not None:
            assert bool(a[[0, 1, 3]].isnan().all()) and torch.equal(a[2:3], b) and not bool(b.isnan().any())
    assert torch.equal(got[4].cpu(), torch.arange(5, dtype=torch.int32)) and torch.equal(got[3][2:3], inner[3]) and torch.equal(got[2][2:3], inner[2])


@pytest.mark.parametrize("n,hq,hkv,bs,rows,seen,keys,split", [
    (1, 32, 8, 16, 400, 400, 400, True), (1, 32, 8, 16, 399, 399, 399, False), (33, 32, 8, 16, 1000, 512, 512, False), (1, 32, 1, 16, 1000, 1000, 1000, False),
    (1, 16, 1, 16, 1000, 1000, 1000, False), (1, 32, 8, 32, 1000, 1000, 1000, False),
    # rows against the longest context
    (8, 32, 8, 16, 4096, 512, 2048, True), (9, 32, 8, 16, 4097, 512, 512, False), (32, 32, 8, 16, 16384, 512, 512, False), (32, 32, 8, 16, 3200, 1100, 1104, True),
    # partial sums of 520 bytes per row, head and 128 keys: 128 MiB of them, and one part more
    (32, 32, 8, 16, 600, 32256, 32256, True), (32, 32, 8, 16, 600, 32257, 32257, False), (32, 32, 8, 16, 600, 512, 131072, False), (1, 32, 8, 16, 600, 512, 131072, True)])
def test_choice_of_split_keys(n, hq, hkv, bs, rows, seen, keys, split):
    assert ops.kept_rows_split(n, hq, hkv, bs, rows, seen, keys) is split


def test_scratch_of_prompt_steps_is_counted(monkeypatch):
    """The cache leaves room for a layer's slabs and the kept rows' splits, beside the slack for the rest."""
    from types import SimpleNamespace

    from src.config import EngineConfig
    from src.engine.llm_engine import plan_kv_blocks
    from src.engine.model_runner import KVPool
    from src.models.presets import get_preset

    free, arch = 1 << 36, get_preset("llama3-8b")
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda dev: (free, free))
    cfg = EngineConfig(max_num_seqs=32, max_num_batched_tokens=4096, gpu_memory_fraction=1.0)
    blocks = plan_kv_blocks(arch, SimpleNamespace(hq=32, hkv=8, inter=14336), cfg, torch.device("cuda"))
    left = free - blocks * KVPool.bytes_per_block(arch.num_layers, 8, cfg.block_size, 128)
    rows = 4096 * (3 * 4096 + 48 * 128 + 3 * 14336) * 2 + 32 * arch.vocab_size * 4
    assert left - rows - (2 << 30) >= 3 * ops.PROMPT_SLAB_BYTES + ops.KEPT_PARTIALS_BYTES
    for m in (129, 256, 257, 1024, 2048):
        for n, k in ((4096, 14336), (8192, 28672), (6144, 4096), (5120, 5120)):
            for residual in (True, False):
                plan = ops.prompt_slab_parts(m, n, k, 256, residual)
                assert plan is None or plan[0] * m * n * 4 <= ops.PROMPT_SLAB_BYTES
