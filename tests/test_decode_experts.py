"""The host side of the decode steps' expert products (``decode_experts``), with a stand-in for the kernels: which products are
launched, with assertions off too, and that every tile that it asks for exists."""

import os
import subprocess
import sys

import pytest
import torch

from src import ops
from src.ops import mix

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

COUNT = """
import torch
from src.ops import mix

class Kernels:
    ran = []
    def gemm_decode_ids(self, y, x, w, *rest):
        self.ran.append(tuple(w.shape))
        return True

x, ids = torch.zeros(4, 256, dtype=torch.bfloat16), torch.zeros(4, 2, dtype=torch.int32)
w13, w2 = torch.zeros(3, 1024, 256, dtype=torch.bfloat16), torch.zeros(3, 256, 512, dtype=torch.bfloat16)
mix.decode_experts(Kernels(), x, w13, w2, ids, 2, 4, mix.MOE_SILU)
print(len(Kernels.ran), Kernels.ran == [(3, 1024, 256), (3, 256, 512)])
"""


@pytest.mark.parametrize("flags", [[], ["-O"]])
def test_both_products_run_without_assertions_too(flags):
    env = dict(os.environ, PYTHONPATH=ROOT)
    out = subprocess.run([sys.executable, *flags, "-c", COUNT], cwd=ROOT, env=env, capture_output=True, text=True, timeout=300)
    assert out.stdout.split() == ["2", "True"], out.stdout + out.stderr


def test_a_second_product_that_does_not_run_is_an_error():
    class Kernels:
        def gemm_decode_ids(self, y, x, w, *rest):
            return w.shape[1] == 1024   # the first one only

    x, ids = torch.zeros(4, 256, dtype=torch.bfloat16), torch.zeros(4, 2, dtype=torch.int32)
    w13, w2 = torch.zeros(3, 1024, 256, dtype=torch.bfloat16), torch.zeros(3, 256, 512, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError):
        mix.decode_experts(Kernels(), x, w13, w2, ids, 2, 4, mix.MOE_SILU)


@pytest.mark.parametrize("t", [1, 16, 32, 33, 64, 65, 128])
def test_every_tile_that_is_asked_for_exists(t):
    """The kernel takes the images of up to 32, 64 or 128 rows."""
    image = 32 if t <= 32 else 64 if t <= 64 else 128
    for n in (32, 48, 64, 96, 128, 192, 1024, 4096):
        for k in (32, 64, 128, 192, 256, 320, 2048):
            for gate in (False, True):
                for pairs in (1, 2, 8, 256):
                    tile = mix._ids_tile(n, k, gate, t, pairs)
                    if tile is not None:
                        assert n % (tile[0] // 2 if gate else tile[0]) == 0 and k % tile[1] == 0
                        assert ops.gd_tile_valid(*tile, image)
