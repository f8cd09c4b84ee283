"""RMSNorm rows that are not whole, aligned 16-byte packs: widths around the packs and the launch shapes, and
operands off 16-byte boundaries, in every mode, forward and backward, under Popcorn's rule against the oracle."""

import pytest
import torch

from oracle import reference as O
from popcorn_amd import _lib, impls
from popcorn_amd.compat import references as R
from tests._parity import gauge_ok, seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _device():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def _check(x, w, b, dy, what):
    """rms_norm of host tensors x, w, b placed on the device as they lie."""
    n64 = [None if t is None else t.double().numpy() for t in (x, w, b, dy)]
    y64 = O.rms_norm(n64[0], n64[1], n64[2], 1e-6)
    dx64, dw64, db64 = O.rms_norm_bwd(n64[0], n64[1], n64[3], 1e-6)
    ref = [t.clone().requires_grad_() for t in (x, w, b) if t is not None]
    yr = R.rms_norm(*ref, eps=1e-6)
    gr = torch.autograd.grad(yr, ref, dy)
    dev = [_place(t).requires_grad_() for t in (x, w, b) if t is not None]
    y = impls.rms_norm(*dev, eps=1e-6)
    got = torch.autograd.grad(y, dev, _place(dy))
    gauge_ok(y, y64, yr, x.dtype, f"y {what}")
    for name, g, t, r in zip(("dx", "dw", "db"), got, (dx64, dw64, db64), gr):
        gauge_ok(g, t, r, x.dtype, f"{name} {what}")


OFFSET = 0


def _place(t):
    """t on the device, OFFSET elements into its buffer."""
    flat = torch.empty(t.numel() + 8, dtype=t.dtype, device=DEV)
    view = flat[OFFSET:OFFSET + t.numel()].view(t.shape)
    view.copy_(t)
    return view.detach()


# one element past, one short of, and a full pack; around one wave's 64, 128 and 256 packs and the block
# shapes' ends (4-byte packs hold 4 elements, 2-byte packs 8)
@pytest.mark.parametrize("dtype,cols", [
    (torch.float32, c) for c in (4, 5, 7, 255, 257, 1023, 1025, 2049, 4099, 16387)] + [
    (torch.bfloat16, c) for c in (8, 9, 15, 511, 513, 2047, 2049, 4097, 8199, 32771)] + [
    (torch.float16, c) for c in (9, 1001, 2050)], ids=str)
@pytest.mark.parametrize("bias", [False, True], ids=["plain", "bias"])
def test_ragged_widths(dtype, cols, bias):
    rows = 9 if cols > 3000 else 301
    x, w, dy = seeded((rows, cols), 1, dtype), seeded((cols,), 2, dtype), seeded((rows, cols), 3, dtype)
    _check(x, w, seeded((cols,), 4, dtype) if bias else None, dy, f"{dtype} cols {cols}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("cols", [64, 1000, 4096])
@pytest.mark.parametrize("offset", [1, 3])
def test_operands_off_16_byte_boundaries(dtype, cols, offset, monkeypatch):
    monkeypatch.setattr("tests.test_gpu_rmsnorm_ragged.OFFSET", offset)
    x, w, dy = seeded((37, cols), 5, dtype), seeded((cols,), 6, dtype), seeded((37, cols), 7, dtype)
    _check(x, w, None, dy, f"offset {offset}")


@pytest.mark.parametrize("dtype,wdtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
                                          (torch.float16, torch.float32)], ids=str)
@pytest.mark.parametrize("cols", [13, 1537, 2051])
def test_ragged_residual_add(dtype, wdtype, cols):
    x, r, w = seeded((130, cols), 1, dtype), seeded((130, cols), 2, dtype), seeded((cols,), 3, wdtype)
    dy, ds = seeded((130, cols), 4, wdtype), seeded((130, cols), 5, dtype)
    leaves = [t.clone().requires_grad_() for t in (x, r, w)]
    ref = R.add_rms_norm(*leaves, 1e-6, 1.0)
    gref = torch.autograd.grad(ref, leaves, (dy, ds))
    truth = [t.double().requires_grad_() for t in (x, r, w)]
    s64 = (x + r).double()  # the sum is rounded to the inputs' type before it is normalised
    s64 = truth[0] + truth[1] + (s64 - truth[0].detach() - truth[1].detach())
    y64 = s64 * torch.rsqrt(s64.square().mean(-1, keepdim=True) + 1e-6) * (truth[2] + 1.0)
    g64 = torch.autograd.grad((y64, s64), truth, (dy.double(), ds.double()))
    dev = [t.to(DEV).requires_grad_() for t in (x, r, w)]
    y, s = impls.add_rms_norm(*dev, 1e-6, 1.0)
    assert torch.equal(s.cpu(), x + r)
    got = torch.autograd.grad((y, s), dev, (dy.to(DEV), ds.to(DEV)))
    gauge_ok(y, y64.detach().numpy(), ref[0], wdtype, "y")
    for name, g, t, q in zip(("dx", "dr", "dw"), got, g64, gref):
        gauge_ok(g, t.numpy(), q, g.dtype, f"{name} cols {cols}")


# one wave to a row and a block to a row, the last pack overlapping by one element and by all but one, whole
# packs, rows narrower than a pack and wider than the row kernels take
@pytest.mark.parametrize("dtype,cols", [
    (torch.float32, c) for c in (3, 5, 7, 1024, 1025, 1537, 4099, 70001)] + [
    (torch.bfloat16, c) for c in (9, 15, 2041, 2049, 4097, 8199, 4096)] + [(torch.float16, 1001)], ids=str)
@pytest.mark.parametrize("into", ["x", "residual"])
def test_add_rms_norm_into_its_own_residual_stream(dtype, cols, into):
    """s written over x or over residual: y, s and rstd are those of a call with buffers of their own."""
    rows, lib = 67, _lib.load()
    x, r, w = seeded((rows, cols), 1, dtype).to(DEV), seeded((rows, cols), 2, dtype).to(DEV), seeded((cols,), 3, dtype).to(DEV)

    def call(x, r, s):
        y, rstd = torch.empty_like(x), torch.empty(rows, device=DEV)
        _lib.check(lib.pk_add_rmsnorm_fwd(x.data_ptr(), r.data_ptr(), w.data_ptr(), y.data_ptr(), s.data_ptr(),
                                          rstd.data_ptr(), rows, cols, 1e-6, 1.0, _lib.dtype_code(dtype),
                                          _lib.dtype_code(dtype), _lib.stream_handle(x.device)))
        return y, s, rstd

    want = call(x, r, torch.empty_like(x))
    mine = {"x": x.clone(), "residual": r.clone()}
    for a, b in zip(call(mine["x"], mine["residual"], mine[into]), want):
        assert torch.equal(a, b)
