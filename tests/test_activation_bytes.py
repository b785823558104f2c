"""What the engine sets aside for a prompt step's activations holds the scratch of the delta rule, which grows with its rows."""

import json

import pytest
import torch

from src.ops import seq


def _model(tmp_path, family):
    if family == "fekolorn":
        from tests.test_fekolorn import CONFIGS
    else:
        from tests.test_rerozen import CONFIGS
    from src.models.fekolorn import GatedDeltaSpec
    from src.models.registry import resolve

    config = CONFIGS["std"]()
    (tmp_path / "config.json").write_text(json.dumps(config))
    _, arch, cls = resolve(str(tmp_path))
    mixers = [getattr(l.mixer, "right", l.mixer) for l in arch.layers]
    return cls(arch, "cpu", dtype=torch.float32), max(m.heads for m in mixers if isinstance(m, GatedDeltaSpec))


@pytest.mark.parametrize("family", ["fekolorn", "rerozen"])
def test_scratch_of_the_delta_rule_is_counted(tmp_path, family):
    """Results are so many bytes a row; the scratch is none for one row."""
    model, heads = _model(tmp_path, family)
    rest = lambda t: model.activation_bytes(t) - (1 << 30) - seq.gated_delta_work_bytes(t, heads)
    assert all(rest(t) == t * rest(1) for t in (9, 100, 4096, 16384))


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[16] * 8, [9] * 20, [17] * 9, [1000, 1, 1, 30], [1] * 8, [4096]])
def test_scratch_is_no_more_than_counted(cuda, lens):
    H, D, T, S = 4, 128, sum(lens), len(lens)
    rag = seq.Ragged(torch.cat([torch.arange(n) for n in lens]).to(cuda), torch.tensor([0] + lens).cumsum(0).int().to(cuda), torch.arange(S).int().to(cuda))
    qkv, bg, gate = torch.randn(T, 3 * H * D, device=cuda) * 0.05, torch.rand(T, 2 * H, device=cuda), torch.randn(T, H * D, device=cuda).bfloat16()
    state, norm, out = torch.zeros(S, H, D, D, device=cuda), torch.ones(D, device=cuda), torch.empty(T, H * D, device=cuda).bfloat16()
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    seq.gated_delta(qkv, bg, gate, norm, 1e-6, state, H, H, D, D, rag, out=out)
    took = torch.cuda.max_memory_allocated() - before
    most = seq.gated_delta_work_bytes(T, H)
    assert took <= (most + 511) // 512 * 512 and (took > 0 or max(lens) == 1)
