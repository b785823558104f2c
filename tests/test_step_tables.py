"""Prompt steps hand attention block tables as wide as their longest context, however long a sequence the model may have; decode steps
hand the whole width. On the GPU: the kernel that runs depends on the columns that a step may use and not on the table's stride."""

import pytest
import torch

from src.models.llama import AttnMetadata
from tests import test_datatar, test_fekolorn


def test_columns():
    bt = torch.zeros(3, 64, dtype=torch.int32)
    meta = lambda prefill, ctx: AttnMetadata(is_prefill=prefill, slot_mapping=bt, block_tables=bt, ctx_lens=bt, max_ctx=ctx)
    assert meta(True, 33).step_tables(16).shape == (3, 3) and meta(True, 32).step_tables(16).shape == (3, 2)
    assert meta(True, 33).step_tables(16).stride(0) == 64
    assert meta(True, 0).step_tables(16) is bt and meta(False, 33).step_tables(16) is bt


@pytest.mark.parametrize("family", ["fekolorn", "datatar"])
def test_engine_hands_over_what_the_step_holds(tmp_path, monkeypatch, family):
    from src.ops import mix, seq
    from src.preproc import SamplingParams

    if family == "fekolorn":
        tests, cfg = test_fekolorn, test_fekolorn.std_config(vocab=48)
        wts, mod, name = tests.orc.make_weights(cfg, seed=1), seq, "sink_attn"
    else:
        tests = test_datatar
        cfg = tests.orc.make_config([(tests.orc.mixer_cfg(), tests.orc.dense_cfg())], vocab=48)
        wts, mod, name = tests.orc.make_weights(cfg, seed=1), mix, "latent_attn"
    eng = tests.make_engine(tmp_path, cfg, wts, "cpu", torch.float32, max_tokens=512, max_seqs=3, mixed_batching="auto")
    eng.eos_token_id = None
    inner, seen = getattr(mod, name), []

    def record(*args, **kw):
        tables = next(a for a in args if torch.is_tensor(a) and a.dtype == torch.int32 and a.dim() == 2)
        ctx = next(a for a in args if torch.is_tensor(a) and a.dtype == torch.int32 and a.dim() == 1 and a.numel() == tables.shape[0])
        cu = next((a for a in args if torch.is_tensor(a) and a.dtype == torch.int32 and a.dim() == 1 and a.numel() == tables.shape[0] + 1), None)
        seen.append((tables.shape[1], int(ctx.max()), cu is not None))
        return inner(*args, **kw)

    monkeypatch.setattr(mod, name, record)
    eng.generate([tests.tokens_for(cfg, n, 20 + n) for n in (5, 23, 40)], SamplingParams(max_tokens=3))
    prompts = [(w, c) for w, c, prompt in seen if prompt]
    assert prompts and all(w == -(-c // 16) for w, c in prompts)
    assert all(w == 32 for w, _, prompt in seen if not prompt)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,past", [((300,), 0), ((128,) * 8, 0), ((200, 190), 0), ((20,), 300), ((60,) * 32, 0)])
def test_unused_columns_change_nothing(cuda, monkeypatch, lens, past):
    from src.ops import mix, seq

    torch.manual_seed(len(lens))
    kern, forms, bs, heads, groups, dim, vdim = mix._kern(), [], 16, 16, 4, 128, 128
    S, T, need = len(lens), sum(lens), -(-(max(lens) + past) // bs)
    wide = torch.randint(0, 3 * need, (S, 256), device=cuda, dtype=torch.int32)   # tables of 4096 tokens
    cu = torch.tensor([0, *lens], device=cuda).cumsum(0).int()
    pos = torch.cat([torch.arange(n) + past for n in lens]).to(cuda)
    ctx = torch.tensor([n + past for n in lens], device=cuda, dtype=torch.int32)
    meta = AttnMetadata(is_prefill=True, slot_mapping=pos, block_tables=wide, ctx_lens=ctx, cu_q=cu, max_q_len=max(lens), max_ctx=max(lens) + past)
    q, cache = torch.randn(T, heads * dim, device=cuda).bfloat16(), torch.randn(3 * need, bs, groups * (dim + vdim), device=cuda).bfloat16()
    q_lat, ql = torch.randn(heads, T, 256, device=cuda).bfloat16(), torch.randn(T, heads * 128, device=cuda).bfloat16()
    lat, inv, sink = torch.randn(3 * need, bs, 288, device=cuda).bfloat16(), mix.rope_inv_freq(10000.0, 32, cuda), torch.randn(heads, device=cuda)

    class Recording:
        def __getattr__(self, name):
            fn = getattr(kern, name)
            return (lambda *a: forms.append(fn(*a))) if name in ("sink_attn", "latent_attn") else fn

    monkeypatch.setattr(seq, "_kern", lambda: Recording())
    monkeypatch.setattr(mix, "_kern", lambda: Recording())
    outs = []
    for tables in (meta.step_tables(bs), wide[:, :need].contiguous()):
        outs.append((seq.sink_attn(q, cache, tables, cu, ctx, pos, None, None, max(lens), heads, groups, dim, vdim, 0, dim ** -0.5),
                     mix.latent_attn(q_lat, ql, 96, lat, tables, cu, ctx, pos, sink, max(lens), 0, 128 ** -0.5, 32, inv)))
    assert forms[:2] == forms[2:] and torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    assert past > 0 or forms[:2] == ["rows", "rows"]
