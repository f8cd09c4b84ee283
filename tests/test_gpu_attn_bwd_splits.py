"""Backward grids of few blocks: dq with its keys split over wave groups, and dk/dv with their query tiles
split into runs (some empty: late key tiles of a causal call have few), against the same sequence in a batch
that fills the device and takes neither.

Only the order of fp32 sums differs, of products rounded alike: between two orders of n tiles of 32 terms a
sum moves by at most n units of fp32 of the sum of its terms' magnitudes, and the result by one unit of its
type; the forward's O, split or not, likewise, whose difference reaches dS through D = rowsum(dO O). Compared
in the 2-norm, that is a unit of the type for each of the three.
"""

import numpy as np
import pytest
import torch

from oracle import reference as O
from popcorn_amd import _lib, impls
from tests._parity import seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"
ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


@pytest.fixture(scope="module", autouse=True)
def _device():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def _grads(q, k, v, do, causal):
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    return torch.autograd.grad(impls.attn(*leaves, causal), leaves, do)


# 2 and 4 runs of query tiles (at these sizes the same number with the mask and without), ragged ends, groups that
# split their heads too, every row layout; `heads` and `runs` are what 256 CUs get. The last two have a dq grid of
# more than one and up to two blocks per CU, split from 96 and, up to 64 dims, 192 key tiles on
@pytest.mark.parametrize("s,hq,hkv,d,dtype,causal,heads,runs", [
    (2048, 4, 4, 64, torch.bfloat16, True, 1, 2),
    (2049, 2, 1, 128, torch.float16, True, 2, 2),
    (4097, 1, 1, 128, torch.bfloat16, True, 1, 4),
    (4100, 2, 2, 32, torch.bfloat16, False, 1, 4),
    (2500, 6, 2, 80, torch.bfloat16, True, 3, 2),
    (2080, 3, 3, 96, torch.float16, False, 1, 2),
    (3100, 16, 16, 128, torch.bfloat16, True, 1, 2),
    (6150, 8, 8, 64, torch.bfloat16, True, 1, 2),
], ids=str)
def test_split_grids_match_a_full_one(s, hq, hkv, d, dtype, causal, heads, runs):
    q, k, v, do = (seeded((1, s, h, d), 7 + i, dtype).to(DEV) for i, h in enumerate((hq, hkv, hkv, hq)))
    lse = -(-2 * hq * s * 4 // 256) * 256
    partials = heads * runs * 2 * s * hkv * (64 if d <= 64 else 128) * 4
    assert _lib.load().pk_attn_bwd_workspace(1, s, hq, hkv, d) == lse + partials
    copies = 512 // (hkv * (s // 128)) + 1
    got = _grads(q, k, v, do, causal)
    want = _grads(*(t.repeat(copies, 1, 1, 1) for t in (q, k, v, do)), causal)
    for name, a, b in zip(("dq", "dk", "dv"), got, want):
        diff = (a.float() - b[:1].float()).norm() / b[:1].float().norm()
        assert diff <= 3 * ULP[dtype], f"{name}: {diff:.2e}"
    if s > 2100:
        return
    group = hq // hkv
    truth = O.attention_bwd(*(t.double().cpu().numpy() for t in (q[:, :, :group], k[:, :, :1], v[:, :, :1], do[:, :, :group])),
                            causal, None)
    for name, a, t in zip(("dq", "dk", "dv"), (got[0][:, :, :group], got[1][:, :, :1], got[2][:, :, :1]), truth):
        err = np.linalg.norm(a.double().cpu().numpy() - t) / np.linalg.norm(t)
        assert err <= 3 * ULP[dtype], f"{name}: {err:.2e}"


def test_split_packed_sequences():
    """Packed sequences under one grid's splits: a long one, short ones (empty runs) and an empty one."""
    cuts = [0, 2100, 2103, 2103, 2300]
    q, k, v, do = (seeded((2300, 2, 64), 3 + i, torch.bfloat16).to(DEV) for i in range(4))
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    o = impls.attn_varlen(*leaves, torch.tensor(cuts, dtype=torch.int32, device=DEV), True)
    got = torch.autograd.grad(o, leaves, do)
    for lo, hi in ((0, 2100), (2100, 2103), (2103, 2300)):
        truth = O.attention_bwd(*(t[lo:hi][None].double().cpu().numpy() for t in (q, k, v, do)), True, None)
        for name, a, t in zip(("dq", "dk", "dv"), got, truth):
            err = np.linalg.norm(a[lo:hi].double().cpu().numpy() - t[0]) / np.linalg.norm(t)
            assert err <= 3 * ULP[torch.bfloat16], f"{name} [{lo}, {hi}): {err:.2e}"
