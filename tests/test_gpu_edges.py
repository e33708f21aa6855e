"""GPU tests at the edges of the kernels' tiles and of their dispatch rules, against the
CPU oracle.  Tolerances as in test_gpu_branches.py (fp32 outputs 1e-5, gradients 1e-4; bf16
2e-2, the oracle fed the bf16-rounded inputs)."""
import math

import pytest
import torch

from nsa import _ops
from test_gpu_branches import _check, _make

pytestmark = pytest.mark.gpu


def _lists(seed, B, G, T, n, nb):
    """n slots a row in any order: random blocks (later ones and repeats among them), -1."""
    g = torch.Generator().manual_seed(seed)
    idx = torch.randint(0, nb, (B, G, T, n), generator=g)
    idx[torch.rand(B, G, T, n, generator=g) < 0.2] = -1
    return idx


# a wave's block bitmaps: 31 / 32 / 33 / 65 blocks (word edges), one to seventeen timesteps a
# wave (1, 2, 3, 4, 15, 20 heads a group), blocks of one, two and three 16-key groups
@pytest.mark.parametrize("hpg,T,lp,n", [(1, 512, 16, 5), (2, 496, 16, 16), (3, 528, 16, 7), (4, 1040, 16, 16),
                                        (15, 130, 48, 3), (20, 131, 32, 64)])
@pytest.mark.parametrize("dtype,dk,dv", [(torch.float32, 64, 64), (torch.bfloat16, 64, 64),
                                         (torch.float32, 192, 128), (torch.bfloat16, 128, 128)])
def test_selection_bitmap_edges(dev, hpg, T, lp, n, dtype, dk, dv):
    B, G = 1, 2
    q, kp, v, do = _make(hpg, B, G * hpg, G, T, T, dk, dv, dtype, dev)
    idx = _lists(hpg + T, B, G, T, n, (T + lp - 1) // lp).to(dev)
    _check(_ops.SELECTION, q, kp, v, do, 1 / math.sqrt(dk), dtype, indices=idx, lprime=lp)
