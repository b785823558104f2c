"""The fused softmax router (one wave selects) against the selection kernel that goes through a token's scores one by one: the same
choices and the same weights to the bit, at the edges of the lanes, with ties, a correction that is -inf or NaN, and every K."""

import pytest
import torch

from src.ops import mix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,K", [(1, 1), (5, 2), (10, 2), (63, 63), (64, 6), (65, 8), (200, 70), (256, 256)])
@pytest.mark.parametrize("corrected", [False, True])
def test_same_bits(cuda, E, K, corrected):
    torch.manual_seed(E + K)
    x = (torch.randn(300, E, device=cuda) * 8).round() / 4       # ties
    eye = torch.eye(E, device=cuda)                              # logits = x exactly, on either path
    corr = torch.randn(E, device=cuda).round() / 8
    if E > 4:
        corr[1], corr[3] = float("-inf"), float("nan")
    args = (eye, K, E, corr if corrected else torch.zeros(E, device=cuda))
    want_w, want_i, _ = mix.route_softmax_topk(x, *args)         # prompt-sized: selection alone
    for a, b in ((0, 256), (256, 300)):
        w, i, _ = mix.route_softmax_topk(x[a:b].contiguous(), *args)
        assert torch.equal(i, want_i[a:b]) and torch.equal(w, want_w[a:b])
