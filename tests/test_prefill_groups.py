"""Which prompt attention steps take two groups of waves per row tile (a rule on the host; the kernel itself is tested on the GPU)."""

import pytest

_C = pytest.importorskip("src._C")


@pytest.mark.parametrize("hq,hkv,seqs,rows,keys,groups", [
    # one turn of 256 compute units: new rows, keys and query heads per key head
    (32, 8, 1, 199, 199, 1), (32, 8, 1, 200, 200, 2), (8, 8, 1, 256, 287, 1), (8, 8, 1, 200, 288, 2), (16, 8, 1, 200, 255, 1), (16, 8, 1, 256, 256, 2),
    (32, 8, 1, 1024, 8000, 2), (32, 1, 1, 1024, 1024, 2), (32, 32, 4, 200, 300, 2), (32, 32, 5, 200, 300, 1),
    # a ninth more: lists of tiles, keys before the step
    (32, 8, 1, 1040, 1040, 2), (32, 8, 1, 1040, 1560, 2), (32, 8, 1, 1040, 1561, 1), (16, 4, 1, 2100, 2100, 2), (24, 24, 1, 1500, 1500, 2), (8, 2, 1, 4500, 4500, 1), (16, 1, 1, 2200, 2200, 1),
    (40, 10, 1, 860, 860, 1), (32, 32, 1, 1150, 1150, 2), (36, 36, 1, 1000, 1000, 1),
    # two turns: eight lists, sixteen of many rows
    (32, 8, 1, 2048, 2560, 2), (32, 8, 1, 2048, 2561, 1), (32, 8, 1, 2049, 2049, 1), (64, 8, 1, 1000, 1000, 2), (16, 4, 2, 1500, 1500, 2), (16, 16, 1, 4096, 4096, 2), (32, 8, 2, 2000, 2000, 1),
    (16, 8, 2, 2000, 2000, 2), (32, 8, 2, 1000, 1000, 1), (16, 4, 3, 1300, 1300, 1), (32, 32, 1, 2048, 2048, 1), (16, 16, 4, 1000, 1000, 1), (8, 8, 8, 1000, 1000, 1), (16, 4, 1, 4096, 4096, 1),
    (16, 1, 1, 3000, 3000, 1), (32, 1, 1, 2048, 2048, 1), (32, 2, 2, 1000, 1000, 1), (64, 2, 1, 1000, 1000, 1), (32, 8, 64, 512, 512, 1)])
def test_groups(hq, hkv, seqs, rows, keys, groups):
    assert _C.attn_prefill_groups(rows, seqs, hq, hkv, keys, 256) == groups


def test_heads_that_make_no_groups():
    assert [_C.attn_prefill_groups(300, 1, hq, hkv, 300, 256) for hq, hkv in ((8, 0), (1, 2), (0, 0))] == [1, 1, 1]
