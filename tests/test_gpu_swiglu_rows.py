"""SwiGLU on rows of a wider tensor, read where they lie: every element's arithmetic is that of the
contiguous call on the same values, so outputs and gradients equal it bit for bit."""

import pytest
import torch

from popcorn_amd import _lib, impls
from tests._parity import seeded

DEV = "cuda"


def _views(kind, rows, cols, dtype):
    """a and b [.., cols] as different programs have them."""
    if kind == "halves":
        return seeded((rows, 2 * cols), 3, dtype).to(DEV).chunk(2, dim=-1)
    if kind == "halves3d":
        return seeded((2, rows, 2 * cols), 3, dtype).to(DEV).chunk(2, dim=-1)
    if kind == "odd_offset":  # rows of one width, starting one element into a buffer, beside contiguous ones
        flat = seeded((rows * (cols + 3) + 1,), 4, dtype).to(DEV)
        return flat[1:].view(rows, cols + 3)[:, :cols], seeded((rows, cols), 5, dtype).to(DEV)
    if kind == "expanded":  # one row for all
        return seeded((1, cols), 6, dtype).to(DEV).expand(rows, cols), seeded((rows, cols + 8), 7, dtype).to(DEV)[:, 8:]
    # rows no single stride reaches: copied, as any other layout
    return seeded((3, rows, cols), 8, dtype).to(DEV).transpose(0, 1), seeded((rows, 3, cols + 1), 9, dtype).to(DEV)[..., 1:]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("rows,cols", [(1, 64), (5, 3), (3, 7), (4, 8), (7, 9), (129, 121), (33, 1000), (65, 14336), (2, 15)], ids=str)
@pytest.mark.parametrize("kind", ["halves", "halves3d", "odd_offset", "expanded", "mixed"])
def test_rows_match_the_contiguous_call(kind, rows, cols, dtype):
    a, b = _views(kind, rows, cols, dtype)
    dy = seeded(tuple(a.shape), 11, dtype).to(DEV)
    with torch.no_grad():
        y = impls.swiglu(a, b)
        want = impls.swiglu(a.contiguous(), b.contiguous())
    assert y.is_contiguous() and torch.equal(y, want)
    views = [t.detach().requires_grad_() for t in (a, b)]
    packed = [t.detach().contiguous().clone().requires_grad_() for t in (a, b)]
    got = torch.autograd.grad(impls.swiglu(*views), views, dy)
    want = torch.autograd.grad(impls.swiglu(*packed), packed, dy)
    for g, w in zip(got, want):
        assert torch.equal(g, w)


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["native", "python"])
def test_a_projection_overwritten_before_the_backward_is_refused(path, monkeypatch):
    """The halves are read in the backward where they lie: a program that reuses their buffer before gets
    autograd's error, as from torch's own ops, and no gradients of the new values."""
    if path == "python":
        monkeypatch.setattr(_lib, "_native", _lib._ThroughPython())
    for op in (impls.swiglu, lambda a, b: torch.nn.functional.silu(a) * b):
        h = seeded((5, 64), 1, torch.float32).to(DEV).requires_grad_() * 1
        y = op(*h.chunk(2, dim=-1))
        with torch.no_grad():
            h.zero_()
        with pytest.raises(RuntimeError, match="inplace"):
            y.sum().backward()
    # what has to be copied to be read is the call's own
    h = seeded((64, 5), 1, torch.float32).to(DEV).requires_grad_() * 1
    y = impls.swiglu(*h.t().chunk(2, dim=-1))
    with torch.no_grad():
        h.zero_()
    y.sum().backward()


def test_row_strides():
    """Which layouts are rows of one stride (host logic)."""
    x = torch.empty(6, 4, 32)
    assert impls._row_stride(x.chunk(2, -1)[1]) == 32
    assert impls._row_stride(x[:, ::2, :16]) == 64
    assert impls._row_stride(x[:, :1, :8]) == 128
    assert impls._row_stride(x[:1, :1, :8]) == 8
    assert impls._row_stride(x[0, 0].expand(5, 32)) == 0
    for t in (x.transpose(0, 1), x[..., ::2], x[:0], torch.empty(3), torch.empty(())):
        assert impls._row_stride(t) is None


def test_rows_arguments_are_checked_before_any_launch():
    lib = _lib.load()
    fwd, bwd = lib.pk_swiglu_rows_fwd, lib.pk_swiglu_rows_bwd
    assert fwd(None, None, None, 0, 8, 8, 8, _lib.BF16, None) == _lib.OK
    assert fwd(None, None, None, 8, 0, 8, 8, _lib.BF16, None) == _lib.OK
    assert fwd(None, None, None, -1, 8, 8, 8, _lib.BF16, None) == _lib.ERR_INVALID
    assert fwd(None, None, None, 2, 8, 8, 8, _lib.BF16, None) == _lib.ERR_INVALID
    assert fwd(16, 16, 16, 2, 8, -8, 8, _lib.BF16, None) == _lib.ERR_INVALID
    assert fwd(16, 16, 16, 2, 8, 8, 8, 7, None) == _lib.ERR_UNSUPPORTED
    assert bwd(16, 16, 16, 16, None, 2, 8, 8, 8, _lib.BF16, None) == _lib.ERR_INVALID
