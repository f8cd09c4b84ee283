"""The native call path against the same calls made through Python: one set of kernels, so every output and
gradient is equal bit for bit, and what autograd does around them is the same."""

import pytest
import torch

from popcorn_amd import _lib, impls
from tests._parity import seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF, F32 = torch.bfloat16, torch.float32


@pytest.fixture(scope="module", autouse=True)
def _device():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def _t(shape, dtype=BF, seed=0):
    return seeded(shape, seed, dtype).to(DEV)


def _heads_first(b, h, s, d, dtype=BF, seed=0):
    return _t((b, s, h, d), dtype, seed).transpose(1, 2)


# op -> (call over its differentiable inputs, those inputs, other inputs)
CASES = {
    "rms_norm": (lambda x, w: impls.rms_norm(x, w), [_t, (6, 40)], [_t, (40,)]),
    "rms_norm_bias": (lambda x, w, b: impls.rms_norm(x, w, b, 1e-5), [_t, (2, 3, 33)], [_t, (33,), F32], [_t, (33,), F32]),
    "add_rms_norm": (lambda x, r, w: impls.add_rms_norm(x, r, w, 1e-6, 1.0), [_t, (6, 40)], [_t, (6, 40)], [_t, (40,)]),
    "swiglu": (lambda x: impls.swiglu(*x.chunk(2, -1)), [_t, (2, 5, 30)]),
    "swiglu_scalar": (impls.swiglu, [_t, ()], [_t, ()]),
    "rotary": (lambda x: impls.rotary_embedding(x, _t((7, 8), F32, 3), _t((7, 8), F32, 4), True), [_t, (2, 7, 3, 32)]),
    "rope": (lambda q, k: impls.rope(q, k, _t((1, 7, 32), F32, 3), _t((1, 7, 32), F32, 4)), [_heads_first, 2, 4, 7, 32],
             [_heads_first, 2, 1, 7, 32]),
    "qk_norm_rope": (lambda q, k, qw, kw: impls.qk_norm_rope(q, k, qw, kw, _t((2, 7, 32), BF, 3), _t((2, 7, 32), BF, 4)),
                     [_heads_first, 2, 4, 7, 32], [_heads_first, 2, 1, 7, 32], [_t, (32,)], [_t, (32,)]),
    "attn": (lambda q, k, v: impls.attn(q, k, v, True, 0.25), [_t, (2, 37, 4, 64)], [_t, (2, 37, 2, 64)], [_t, (2, 37, 2, 64)]),
    "attn_f32": (lambda q, k, v: impls.attn(q, k, v), [_t, (1, 37, 4, 40), F32], [_t, (1, 37, 2, 40), F32],
                 [_t, (1, 37, 2, 40), F32]),
    "attn_varlen": (lambda q, k, v: impls.attn_varlen(q, k, v, torch.tensor([0, 5, 5, 37]), True), [_t, (37, 4, 64)],
                    [_t, (37, 2, 64)], [_t, (37, 2, 64)]),
}


def _leaves(specs):
    return [make(*args).detach().requires_grad_() for make, *args in specs]


def _run(call, leaves):
    outs = call(*leaves)
    outs = outs if isinstance(outs, tuple) else (outs,)
    dys = [torch.ones_like(o) * (i + 1) for i, o in enumerate(outs)]
    return [o.detach() for o in outs], torch.autograd.grad(outs, leaves, dys)


@pytest.fixture
def through_python(monkeypatch):
    def switch():
        monkeypatch.setattr(_lib, "_native", _lib._ThroughPython())

    assert not isinstance(_lib.native(), _lib._ThroughPython), "the extension module was not built for this torch"
    return switch


@pytest.mark.parametrize("name", list(CASES))
def test_native_calls_match_the_python_path(name, through_python):
    call, *specs = CASES[name]
    got = _run(call, _leaves(specs))
    with torch.no_grad():
        plain = call(*_leaves(specs))
    with torch.autograd.graph.save_on_cpu():  # hooks: the saved tensors come back as other tensors
        hooked = _run(call, _leaves(specs))
    through_python()
    want = _run(call, _leaves(specs))
    for mine in (got, hooked):
        for a, b in zip(mine[0] + list(mine[1]), want[0] + list(want[1])):
            assert a.dtype == b.dtype and torch.equal(a, b)
    for a, b in zip(plain if isinstance(plain, tuple) else (plain,), want[0]):
        assert torch.equal(a, b) and not a.requires_grad


@pytest.mark.parametrize("name", ["add_rms_norm", "rope", "qk_norm_rope"])
@pytest.mark.parametrize("used", [0, 1])
def test_a_gradient_through_one_output_only(name, used, through_python):
    call, *specs = CASES[name]

    def grads():
        leaves = _leaves(specs)
        out = call(*leaves)[used]
        return torch.autograd.grad(out, leaves, torch.ones_like(out), allow_unused=True)

    got = grads()
    through_python()
    for a, b in zip(got, grads()):
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b))


def test_autograd_refuses_what_it_refused(through_python):
    """A changed input, a second backward and the function transforms, natively and through Python."""
    for switch in (lambda: None, through_python):
        switch()
        x, w = _t((4, 64)).requires_grad_(), _t((64,)).requires_grad_()
        h = x * 1
        y = impls.rms_norm(h, w)
        h.add_(1)
        with pytest.raises(RuntimeError, match="inplace"):
            y.sum().backward()
        y = impls.rms_norm(x, w)
        y.sum().backward()
        with pytest.raises(RuntimeError, match="second time"):
            y.sum().backward()
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda t: impls.rms_norm(t, w).sum())(x.detach())
        with pytest.raises(Exception):
            torch.func.vmap(lambda t: impls.rms_norm(t, w))(x.detach()[None])
        with pytest.raises(TypeError, match="not supported"):
            impls.rms_norm(_t((4, 64), F32), w)
        with pytest.raises(ValueError, match="several devices"):
            impls.rms_norm(x, w.detach().cpu())


def test_layouts_that_need_a_copy_and_subclasses_are_left_to_python():
    native = _lib.native()
    x, w = _t((8, 64)), _t((64,))
    assert native.rms_norm(x.t().contiguous().t(), w, None, 1e-6) is NotImplemented
    assert native.rms_norm(x[:0], w, None, 1e-6) is NotImplemented
    assert native.rms_norm(x, w, None, 1) is NotImplemented  # an integer eps: Python converts it
    assert native.rms_norm(x.as_subclass(type("Sub", (torch.Tensor,), {})), w, None, 1e-6) is NotImplemented
    assert native.attn(*(_t((1, 9, 2, 64))[..., :60] for _ in range(3)), False, None) is NotImplemented
    assert torch.equal(impls.rms_norm(x.t().contiguous().t(), w), impls.rms_norm(x, w))


def test_a_torch_function_mode_sees_the_calls_inside():
    """As it does through Python; the mode of a default device, which changes nothing here, does not matter."""

    class Seen(torch.overrides.TorchFunctionMode):
        names = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.names.append(getattr(func, "__name__", str(func)))
            return func(*args, **(kwargs or {}))

    x, w = _t((4, 64)), _t((64,))
    want = impls.rms_norm(x, w)
    with Seen():
        assert torch.equal(impls.rms_norm(x, w), want)
    assert "empty" in Seen.names
    with torch.device("cpu"):
        assert torch.equal(_lib.native().rms_norm(x, w, None, 1e-6), want)
        with Seen():
            assert _lib.native().rms_norm(x, w, None, 1e-6) is NotImplemented
    assert torch.equal(_lib.native().rms_norm(x, w, None, 1e-6), want)


def test_tangents_are_refused_as_before(through_python):
    """Forward-mode AD: no op has a jvp, so a dual input is refused and not read past its tangent."""
    fwad = torch.autograd.forward_ad
    x, w = _t((4, 64)), _t((64,))
    for switch in (lambda: None, through_python):
        switch()
        with fwad.dual_level():
            dual = fwad.make_dual(x, torch.ones_like(x))
            if switch is not through_python:
                assert _lib.native().rms_norm(dual, w, None, 1e-6) is NotImplemented
            with pytest.raises(NotImplementedError):
                impls.rms_norm(dual.requires_grad_(), w)
        assert torch.equal(impls.rms_norm(x, w), impls.rms_norm(x.clone(), w))


def test_a_traced_call_stays_in_python(monkeypatch):
    """Where the tracer is at work the native path is not offered the call at all."""

    class Refuses:
        def __getattr__(self, name):
            raise AssertionError("the native path was offered a traced call")

    x, w = _t((4, 64)), _t((64,))
    want = impls.rms_norm(x, w)
    monkeypatch.setattr(impls, "_compiling", lambda: True)
    monkeypatch.setattr(_lib, "_native", Refuses())
    assert torch.equal(impls.rms_norm(x, w), want)


@pytest.mark.parametrize("name", ["rms_norm", "swiglu", "attn"])
def test_calls_go_on_the_current_stream(name):
    """Forward and backward on a stream of their own, after work there that the inputs wait for."""
    call, *specs = CASES[name]
    want = _run(call, _leaves(specs))
    side = torch.cuda.Stream()
    ready = _leaves(specs)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        held = torch.randn(4096, 4096, device=DEV)
        for _ in range(20):
            held = held @ held * 1e-4  # some milliseconds ahead of the copies
        late = [torch.zeros_like(t) for t in ready]
        for dst, src in zip(late, ready):
            dst.copy_(src.detach())
        got = _run(call, [t.requires_grad_() for t in late])
    side.synchronize()
    for a, b in zip(got[0] + list(got[1]), want[0] + list(want[1])):
        assert torch.equal(a, b)
