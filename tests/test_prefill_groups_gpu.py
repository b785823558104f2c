"""Prompt attention in two groups of waves per workgroup (attention.hip, steps of few row tiles) against fp32 attention.

Weights and results are rounded to bf16 once each (2^-9 of each value, at random): the 2-norm of the difference is within 2^-8 of that of the result, and
no value is further off than 2^-6 of the rows' largest scale."""

import math

import pytest
import torch

from src import ops
from src.ops import reference as ref

pytestmark = pytest.mark.gpu


# new tokens and lengths: one stage for the first group alone, odd and even numbers of stages, a row of one key beside long ones, keys before the step, more than one turn of
# row tiles with 8 key heads
CASES = [([200], [200]), ([257], [257]), ([1, 320, 33], [1, 320, 33]), ([288, 5], [1000, 37]), ([1000], [1000]), ([1025], [1537]), ([1040], [1040]), ([1500], [1500])]
HEADS = [(8, 4), (4, 1), (1, 8), (1, 32)]


def _groups(qlens, ctxs, hkv, g):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    return ops._kern().attn_prefill_groups(max(qlens), len(qlens), hkv * g, hkv, (max(ctxs) + 15) // 16 * 16, cus)


def test_cases_take_two_groups():
    """All with several heads per key head but the one behind many keys beyond a turn; from 288 keys on with one."""
    taken = {h: [c for c in CASES if _groups(*c, *h) == 2] for h in HEADS}
    assert taken[8, 4] == CASES[:5] + CASES[6:] and taken[4, 1] == CASES[2:] and taken[1, 8] == CASES and taken[1, 32] == CASES[:5]


@pytest.mark.parametrize("qlens,ctxs", CASES)
@pytest.mark.parametrize("hkv,g", HEADS)
def test_groups(qlens, ctxs, hkv, g):
    hq, t, blocks = hkv * g, sum(qlens), [(c + 15) // 16 for c in ctxs]
    rng = torch.Generator(device="cuda").manual_seed(0)
    kc, vc = (torch.randn(sum(blocks), hkv, 16, 128, generator=rng, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(t, hq * 128, generator=rng, device="cuda").bfloat16()
    perm = torch.randperm(sum(blocks), generator=rng, device="cuda").int()
    bt = torch.zeros(len(qlens), max(blocks), dtype=torch.int32, device="cuda")
    at = 0
    for i, n in enumerate(blocks):
        bt[i, :n] = perm[at: at + n]
        at += n
    cu = torch.tensor([0] + qlens).cumsum(0).int().cuda()
    ctx = torch.tensor(ctxs, dtype=torch.int32, device="cuda")
    scale = 1 / math.sqrt(128)
    out = ops.attn_prefill(q, kc, vc, bt, cu, ctx, max(qlens), hq, hkv, scale).float()
    want = ref.attention(q, kc, vc, bt, cu, ctx, hq, hkv, scale).reshape(t, -1).float()
    assert float((out - want).norm() / want.norm()) < 2.0 ** -8
    assert float((out - want).abs().max() / want.abs().max()) < 2.0 ** -6
