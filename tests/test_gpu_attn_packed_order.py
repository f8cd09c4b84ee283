"""Packed sequences whose tiles the blocks find among all the sequences' tiles: every sequence's rows equal
the dense call's on that sequence alone, bit for bit (a tile's arithmetic does not depend on which block runs
it; dk and dv of grouped heads are left out, since how they are split over q heads follows the whole grid)."""

import random

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


def _lengths(seqs, seed):
    """Empty and one-token sequences, whole and ragged tiles, ties, one long sequence somewhere."""
    rng = random.Random(seed)
    lens = [rng.choice((0, 1, 31, 32, 33, 127, 128, 129, 160)) for _ in range(seqs)]
    lens[rng.randrange(seqs)] = 321
    return lens


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("hq,hkv,d", [(8, 8, 64), (3, 3, 128), (32, 8, 64), (6, 2, 96), (4, 4, 192)], ids=str)
@pytest.mark.parametrize("seqs", [2, 23, 64, 65])
def test_every_sequence_matches_its_dense_call(seqs, hq, hkv, d, causal):
    lens = _lengths(seqs, seqs + hq)
    cuts = [0]
    for n in lens:
        cuts.append(cuts[-1] + n)
    total = cuts[-1]
    q, k, v, do = (seeded((total, h, d), 3 + i, torch.bfloat16).to(DEV) for i, h in enumerate((hq, hkv, hkv, hq)))
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    o = impls.attn_varlen(*leaves, torch.tensor(cuts, dtype=torch.int32, device=DEV), causal)
    grads = torch.autograd.grad(o, leaves, do)
    for lo, hi in zip(cuts, cuts[1:]):
        if lo == hi:
            continue
        seg = [t[lo:hi][None].clone().requires_grad_() for t in (q, k, v)]
        want = impls.attn(*seg, causal)
        want_grads = torch.autograd.grad(want, seg, do[lo:hi][None])
        assert torch.equal(o[lo:hi], want[0]), (lo, hi)
        for g, w in list(zip(grads, want_grads))[: 3 if hq == hkv else 1]:
            assert torch.equal(g[lo:hi], w[0]), (lo, hi)
