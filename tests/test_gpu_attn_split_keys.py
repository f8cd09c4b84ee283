"""Attention forward calls of few blocks and long rows, whose keys are split over the groups of a wider
block, against the unsplit kernel on the same rows and the float64 oracle.

The unsplit result of the same rows comes from a batch of enough copies of the sequence that the grid
fills the device. Both forms add the same fp32 products of the same rounded P; only the order of the sum
over key tiles differs, so with at most n tiles a row's outputs differ by at most about n fp32 roundings of
its largest partial sum (bounded by sum(p |v|) / l <= max |v|), plus one rounding of the output.
"""

import numpy as np
import pytest
import torch

from oracle import reference as O
from popcorn_amd import impls
from tests._parity import seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"
ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


@pytest.fixture(scope="module", autouse=True)
def _device():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def _inputs(s, hq, hkv, d, dtype, seed):
    return (seeded((1, s, hq, d), seed, dtype), seeded((1, s, hkv, d), seed + 1, dtype),
            seeded((1, s, hkv, d), seed + 2, dtype))


# one block per CU: tiles of 32 keys around multiples of the group count (2, 3 and 4 groups), a last tile of one
# key, and rows of every layout
@pytest.mark.parametrize("s,hq,hkv,d,dtype,causal", [
    (1023, 4, 1, 64, torch.bfloat16, True),
    (1025, 6, 2, 64, torch.float16, False),
    (1100, 4, 4, 32, torch.bfloat16, True),
    (1537, 4, 1, 128, torch.bfloat16, False),
    (1568, 2, 1, 128, torch.float16, True),
    (1601, 3, 1, 96, torch.bfloat16, True),
    (1540, 4, 2, 192, torch.bfloat16, False),
    (1537, 2, 2, 256, torch.bfloat16, True),
], ids=str)
def test_split_rows_match_the_unsplit_kernel(s, hq, hkv, d, dtype, causal):
    q, k, v = (t.to(DEV) for t in _inputs(s, hq, hkv, d, dtype, 3 * d))
    with torch.no_grad():
        o, lse = impls.attn_with_lse(q, k, v, causal)
        wide, wide_lse = impls.attn_with_lse(*(t.repeat(_copies(s, hq), 1, 1, 1) for t in (q, k, v)), causal)
    tiles = -(-s // 32)
    bound = v.float().abs().max().item() * (2 * tiles * 2.0**-24 + ULP[dtype])
    assert (o.float() - wide[:1].float()).abs().max().item() <= bound
    # l is a sum of n tiles of positive terms: its relative error moves lse by as much
    assert (lse - wide_lse[:1]).abs().max().item() <= 2 * tiles * 2.0**-24 + 2e-6
    rows = np.array([0, 31, 32, s // 2, s - 1])
    for h in (0, hq - 1):
        qh, kh, vh = (t[0, :, i].double().cpu().numpy() for t, i in ((q, h), (k, h * hkv // hq), (v, h * hkv // hq)))
        o64, lse64 = O.attention_rows(qh, kh, vh, rows, causal)
        assert np.abs(o[0, rows, h].double().cpu().numpy() - o64).max() < 2e-2 * max(1.0, np.abs(o64).max())
        np.testing.assert_allclose(lse[0, h, rows].double().cpu().numpy(), lse64, rtol=0, atol=1e-3)


def _copies(s, hq):
    return 4096 // (hq * (s // 128)) + 1  # more than two blocks per CU at any row group


# one block per CU, of 24 to 31 (up to 64 dims) and 28 to 47 key tiles: split where no log-sum-exp is kept
@pytest.mark.parametrize("s,hq,hkv,d,dtype,causal", [
    (768, 4, 1, 64, torch.bfloat16, True),
    (991, 6, 2, 32, torch.float16, False),
    (896, 4, 4, 128, torch.bfloat16, True),
    (1021, 32, 8, 128, torch.bfloat16, True),
    (1500, 2, 1, 192, torch.bfloat16, True),
    (900, 4, 2, 256, torch.float16, True),
], ids=str)
def test_split_without_a_log_sum_exp(s, hq, hkv, d, dtype, causal):
    """No more than the order of the sum over tiles differs from an unsplit grid, and it does differ (the call
    was split); with a log-sum-exp, as a call that is recorded for a backward has it, not even that."""
    q, k, v = (t.to(DEV) for t in _inputs(s, hq, hkv, d, dtype, 2 * d))
    many = [t.repeat(_copies(s, hq), 1, 1, 1) for t in (q, k, v)]
    with torch.no_grad():
        o, wide = impls.attn(q, k, v, causal), impls.attn(*many, causal)[:1]
        kept = impls.attn_with_lse(q, k, v, causal)[0]
    recorded = impls.attn(q.clone().requires_grad_(), k, v, causal).detach()
    bound = v.float().abs().max().item() * (2 * -(-s // 32) * 2.0**-24 + ULP[dtype])
    assert (o.float() - wide.float()).abs().max().item() <= bound
    assert not torch.equal(o, wide)
    assert torch.equal(kept, wide) and torch.equal(recorded, wide)


# causal grids of 257 to 512 blocks (256 CUs): on either side of the lines of split_keys
@pytest.mark.parametrize("s,hq,hkv,d,split", [
    (2048, 32, 32, 128, False),  # one head to a kv head: from 72 tiles on
    (2304, 26, 26, 128, True),
    (2048, 32, 8, 96, True),  # four heads: from 64
    (2048, 32, 32, 256, False),  # wide rows: up to 384 blocks as above, past them from 128 tiles on
    (2310, 17, 17, 192, True),
    (3072, 21, 21, 192, False),
    (4096, 16, 16, 256, True),
    (6100, 8, 8, 64, False),  # up to 64 dims: from 192
    (6150, 8, 8, 64, True),
], ids=str)
def test_split_at_two_blocks_per_cu(s, hq, hkv, d, split):
    q, k, v = (t.to(DEV) for t in _inputs(s, hq, hkv, d, torch.bfloat16, d + 1))
    with torch.no_grad():
        o = impls.attn(q, k, v, True)
        wide = impls.attn(*(t.repeat(_copies(s, hq), 1, 1, 1) for t in (q, k, v)), True)[:1]
    bound = v.float().abs().max().item() * (2 * -(-s // 32) * 2.0**-24 + ULP[torch.bfloat16])
    assert (o.float() - wide.float()).abs().max().item() <= bound
    assert torch.equal(o, wide) is not split


@pytest.mark.parametrize("d", [64, 128, 256])
def test_split_rows_with_late_large_scores(d):
    """Scores far above the first tile's max send a split block to the exact sweep, as an unsplit one."""
    s = 1600
    q, k, v = (t.float() for t in _inputs(s, 4, 1, d, torch.float32, 5))
    k[:, 700:710] *= 8.0
    q[:, 900:] *= 3.0
    q, k, v = (t.to(torch.bfloat16).to(DEV) for t in (q, k, v))
    with torch.no_grad():
        o, lse = impls.attn_with_lse(q, k, v, True)
    rows = np.array([0, 699, 705, 899, 1000, s - 1])
    for h in (0, 3):
        qh, kh, vh = (t[0, :, i].double().cpu().numpy() for t, i in ((q, h), (k, 0), (v, 0)))
        o64, lse64 = O.attention_rows(qh, kh, vh, rows, True)
        assert np.abs(o[0, rows, h].double().cpu().numpy() - o64).max() < 2e-2 * max(1.0, np.abs(o64).max())
        np.testing.assert_allclose(lse[0, h, rows].double().cpu().numpy(), lse64, rtol=1e-5, atol=1e-3)


def test_split_packed_rows():
    """Packed sequences of one long and some short (and no) tokens: the short ones run masked steps only."""
    cu = [0, 1600, 1600, 1601, 1700]
    q, k, v = (t[0] for t in _inputs(1700, 4, 1, 128, torch.bfloat16, 9))
    with torch.no_grad():
        o, lse = impls.attn_varlen_with_lse(*(t.to(DEV) for t in (q, k, v)), torch.tensor(cu, dtype=torch.int32, device=DEV),
                                            True)
    for lo, hi in ((0, 1600), (1600, 1601), (1601, 1700)):
        rows = np.unique(np.array([0, (hi - lo) // 2, hi - lo - 1]))
        o64, lse64 = O.attention_rows(*(t[lo:hi, h].double().numpy() for t, h in ((q, 3), (k, 0), (v, 0))), rows, True)
        assert np.abs(o[lo:hi, 3].double().cpu().numpy()[rows] - o64).max() < 2e-2 * max(1.0, np.abs(o64).max())
        np.testing.assert_allclose(lse[3, lo:hi].double().cpu().numpy()[rows], lse64, rtol=0, atol=1e-3)
