"""The attention of a prompt step's last layer for its kept rows (one query per sequence, by the decode or the prompt kernel) against the same rows of the
step that keeps every row.

Both round weights and results to bf16 once each, 2^-9 of each value at random, and so do the rotated queries: the 2-norm of the difference is within
2^-7 of that of the result. The last layers' hidden states differ by that and by one bf16 rounding per product, as elsewhere 2e-2."""

from dataclasses import replace

import pytest
import torch

from src import ops
from src.models.llama import AttnMetadata, CausalLM
from src.models.presets import get_preset

pytestmark = pytest.mark.gpu


def _model(hq, hkv):
    # (weights large enough that scores differ by some units, so that positions and keys tell)
    arch = replace(get_preset("llama-mini"), hidden_size=512, num_heads=hq, num_kv_heads=hkv, intermediate_size=512, num_layers=2, vocab_size=1024)
    return CausalLM(arch, "cuda:0", seed=3, init_std=0.06, max_position=4096)


def _last_attention(monkeypatch, m, lens, past, bs, max_ctx, keep):
    """(the kernel of the step's last attention call, its rows, the step's hidden states)"""
    calls = []
    with monkeypatch.context() as mp:
        for name in ("attn_prefill", "attn_decode"):
            mp.setattr(ops, name, lambda *a, f=getattr(ops, name), n=name, **k: calls.append((n, f(*a, **k))) or calls[-1][1])
        g = torch.Generator().manual_seed(1)
        t, s = sum(lens), len(lens)
        blocks = [-(-(n + p) // bs) for n, p in zip(lens, past)]
        tables = torch.zeros(s, max(blocks) + 2, dtype=torch.int32)
        perm, at = torch.randperm(sum(blocks), generator=g).int(), 0
        for i, n in enumerate(blocks):
            tables[i, :n] = perm[at: at + n]
            at += n
        pos = torch.cat([torch.arange(n) + p for n, p in zip(lens, past)])
        seq = torch.repeat_interleave(torch.arange(s), torch.tensor(lens))
        slots = tables[seq, pos // bs].long() * bs + pos % bs
        cu = torch.tensor([0, *lens]).cumsum(0).int()
        pool = torch.randn(m.arch.num_layers, 2, sum(blocks), m.hkv, bs, 128, generator=g).to("cuda", m.dtype)
        ctx = torch.tensor([n + p for n, p in zip(lens, past)], dtype=torch.int32)
        last = (cu[1:] - 1).long().cuda()
        meta = AttnMetadata(True, slots.cuda(), tables.cuda(), ctx.cuda(), cu.cuda(), max(lens), max_ctx=int(ctx.max()) if max_ctx else 0,
                            keep_rows=last if keep else None)
        hidden = m.forward(torch.randint(3, 1000, (t,), generator=g).cuda(), pos.cuda(), meta, pool)
    name, rows = calls[-1]
    return (name, rows, hidden) if keep else (name, rows[last], hidden[last])


DEC, PRO = "attn_decode", "attn_prefill"


@pytest.mark.parametrize("hq,hkv,bs,lens,past,max_ctx,kernel", [
    # either side of 400 keys, known by the new rows or by the longest context alone; tables wider than it
    (8, 2, 16, [399], [0], False, PRO), (8, 2, 16, [400], [0], False, DEC), (8, 2, 16, [150, 30], [249, 0], True, PRO),
    (8, 2, 16, [150, 30], [250, 0], True, DEC), (8, 2, 16, [150, 30], [250, 0], False, PRO),
    # ragged lengths behind cached keys, one new row among them
    (8, 2, 16, [500, 1, 260], [0, 700, 77], True, DEC), (8, 2, 16, [500, 1, 260], [0, 700, 77], False, DEC), (8, 8, 16, [129, 64, 3], [1000, 0, 128], True, DEC),
    # sequences times key heads
    (16, 8, 16, [20] * 31 + [400], [0] * 32, True, DEC), (16, 8, 16, [20] * 32 + [400], [0] * 33, True, PRO),
    # every number of query heads per group; another block size
    (8, 4, 16, [450, 70], [0, 40], True, DEC), (16, 2, 16, [450, 70], [0, 40], True, DEC), (16, 1, 16, [450, 70], [0, 40], True, PRO),
    (32, 1, 16, [450, 70], [0, 40], True, PRO), (8, 2, 32, [450, 70], [0, 40], True, PRO)])
@pytest.mark.parametrize("form", ["library", "slabs", "plain norm"])
def test_kept_rows(monkeypatch, hq, hkv, bs, lens, past, max_ctx, kernel, form):
    """Queries turned by the gather, by the pass that sums the projection's slabs, and without a scale per row."""
    m = _model(hq, hkv)
    monkeypatch.setattr(ops, "prompt_slab_parts", lambda mm, n, k, cus, residual: None if residual or form != "slabs" else ops.slab_parts(mm, n, k, cus))
    m.norms_folded = form != "plain norm"
    name, got, hidden = _last_attention(monkeypatch, m, lens, past, bs, max_ctx, True)
    assert name == kernel and got.shape[0] == hidden.shape[0] == len(lens)
    whole, want, rows = _last_attention(monkeypatch, m, lens, past, bs, max_ctx, False)
    assert whole == PRO
    assert float((got.double() - want.double()).norm() / want.double().norm()) < 2.0 ** -7
    assert float((hidden.double() - rows.double()).norm() / rows.double().norm()) < 2e-2
