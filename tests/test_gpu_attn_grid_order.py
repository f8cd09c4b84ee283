"""Causal grids of between one block per CU and as many as are resident at once run in an order of their own.
Every tile has to be run by some block, and which one does not change its arithmetic: each sequence's outputs
and gradients equal those it has in a batch too large for that order, bit for bit."""

import pytest
import torch

from popcorn_amd import impls
from tests._parity import seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _device():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


# grids of 257 to 1023 blocks of the forward, whole and ragged rounds of 32 per XCD, group counts that are and
# are not a multiple of 8, row groups of 32, 64 and 128, every layout with more than one block per CU
@pytest.mark.parametrize("b,s,heads,d,dtype", [
    (3, 1100, (12, 12), 128, torch.bfloat16),
    (11, 1000, (3, 3), 64, torch.float16),
    (4, 900, (24, 8), 32, torch.bfloat16),
    (5, 1030, (14, 7), 96, torch.bfloat16),
    (13, 257, (16, 4), 128, torch.bfloat16),
    (3, 640, (20, 5), 192, torch.bfloat16),
    (2, 1000, (24, 24), 64, torch.float32),
    (7, 333, (20, 5), 128, torch.float32),
], ids=str)
def test_every_tile_is_run_once(b, s, heads, d, dtype):
    hq, hkv = heads
    q, k, v, do = (seeded((b, s, h, d), 5 + i, dtype).to(DEV) for i, h in enumerate((hq, hkv, hkv, hq)))
    copies = 6  # past the resident blocks of every kernel

    def run(*ts):
        leaves = [t.clone().requires_grad_() for t in ts[:3]]
        o = impls.attn(*leaves, True)
        return (o.detach(), *torch.autograd.grad(o, leaves, ts[3]))

    got = run(q, k, v, do)
    want = run(*(t.repeat(copies, 1, 1, 1) for t in (q, k, v, do)))
    names = ("o", "dq", "dk", "dv") if hq == hkv else ("o", "dq")  # grouped heads: the splits follow the grid
    for name, x, y in zip(names, got, want):
        assert torch.equal(x, y[:b]), name
