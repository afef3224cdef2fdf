"""Refusals of the native host layer (csrc/host_calls.cc) that need no GPU: shape-only tensors that claim to live on one
reach the checks of its functions and nothing behind them."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

BF16, F32 = torch.bfloat16, torch.float32
B, LQ, LK, RQ, RK, H, D = 2, 8, 16, 6, 2, 8, 64


@pytest.fixture
def shapes():
    with FakeTensorMode():
        yield lambda *s, dtype=BF16: torch.empty(s, device="cuda", dtype=dtype)


def _concatenated(new, **changed):
    x = dict(q=new(B, LQ, RQ, H + D), k=new(B, LK, RK, H + D), v=new(B, LK, RK, H + D), heads=H)
    x.update(changed)
    return x["q"], x["k"], x["v"], x["heads"]


CONCATENATED = [
    (AssertionError, lambda new: dict(k=new(B, LK - 1, RK, H + D))),  # fewer tokens than v
    (AssertionError, lambda new: dict(k=new(B, LK, RK - 1, H + D))),
    (AssertionError, lambda new: dict(k=new(B, LK, RK, H + D - 8))),
    (AssertionError, lambda new: dict(k=new(B - 1, LK, RK, H + D))),
    (AssertionError, lambda new: dict(k=new(B - 1, LK, RK, H + D), v=new(B - 1, LK, RK, H + D))),
    (AssertionError, lambda new: dict(v=new(B - 1, LK, RK, H + D))),
    (AssertionError, lambda new: dict(heads=0)),
    (AssertionError, lambda new: dict(heads=-1)),
    (AssertionError, lambda new: dict(heads=H + D)),
    (TypeError, lambda new: dict(k=new(B, LK, RK, H + D, dtype=F32))),
    (TypeError, lambda new: dict(v=new(B, LK, RK, H + D, dtype=F32))),
    (ValueError, lambda new: dict(k=new(B, LK * RK, H + D))),
]


@pytest.mark.parametrize("call", ["tpa", "_tpa_bwd"])
@pytest.mark.parametrize("error,changed", CONCATENATED)
def test_the_operator_and_its_gradient_refuse_operands_that_do_not_fit(shapes, call, error, changed):
    from tpa import tpa

    q, k, v, heads = _concatenated(shapes, **changed(shapes))
    with pytest.raises(error):
        if call == "tpa":
            tpa.tpa(q, k, v, heads)
        else:
            o, l = shapes(B, LQ, H, D), shapes(B, LQ, H, dtype=F32)
            tpa._tpa_bwd(heads, 1.0, False, None, False, False, False, (q, k, v, None, None, o, l), o)


def test_the_gradient_of_one_entry_refuses_them_too(shapes):
    from tpa import tpa

    q, k, v, o, l = shapes(LQ, RQ, H + D), shapes(LK - 1, RK, H + D), shapes(LK, RK, H + D), shapes(LQ, H, D), shapes(LQ, H, dtype=F32)
    with pytest.raises(AssertionError):
        tpa._bwd(q, k, v, None, None, o, l, o, H, 1.0, False, None, False, False, False)


@pytest.mark.parametrize("call", ["tpa_factors", "tpa_decode", "tpa_factors_bwd"])
@pytest.mark.parametrize(
    "changed",
    [
        dict(qb=(B, LQ, RQ - 1, D)), dict(ka=(B, LK - 1, RK, H)), dict(ka=(B, LK, RK, H - 1)), dict(kb=(B, LK, RK - 1, D)),
        dict(va=(B - 1, LK, RK, H)), dict(va=(B, LK, RK - 1, H)), dict(vb=(B - 1, LK, RK, D)), dict(vb=(B, LK + 1, RK, D)),
        dict(grads=4),
    ],
)
def test_the_split_forms_refuse_factors_that_do_not_fit(shapes, call, changed):
    from tpa import tpa

    sizes = dict(qa=(B, LQ, RQ, H), qb=(B, LQ, RQ, D), ka=(B, LK, RK, H), kb=(B, LK, RK, D), va=(B, LK, RK, H), vb=(B, LK, RK, D))
    if "grads" in changed and call != "tpa_factors_bwd":
        pytest.skip("takes no gradient arrays")
    x = [shapes(*{**sizes, **changed}[name]) for name in sizes]
    with pytest.raises(AssertionError):
        if call == "tpa_factors_bwd":
            o, lse = shapes(B, LQ, H, x[5].shape[3]), shapes(B, H, LQ, dtype=F32)
            grads = [shapes(*t.shape, dtype=F32) for t in x]
            if "grads" in changed:
                grads[changed["grads"]] = shapes(B, LK - 1, RK, H, dtype=F32)
            tpa.tpa_factors_bwd(*x, None, None, o, lse, o, grads=grads)
        else:
            getattr(tpa, call)(*x)


@pytest.mark.parametrize("which", [0, 1, 2])
def test_forward_mode_raises_instead_of_dropping_the_tangent(shapes, which):
    import torch.autograd.forward_ad as fwd
    from tpa import tpa

    qkv = [shapes(B, LQ, RQ, H + D), shapes(B, LK, RK, H + D), shapes(B, LK, RK, H + D)]
    with fwd.dual_level(), pytest.raises(NotImplementedError):
        qkv[which] = fwd.make_dual(qkv[which], shapes(*qkv[which].shape))
        tpa.tpa(*qkv, H)


@pytest.mark.parametrize("transform", ["vmap", "grad", "vjp", "jvp"])
def test_function_transforms_are_refused(shapes, transform):
    """The node has no rule for them: an error, never a result that ignores the transform."""
    from tpa import tpa

    q, k, v = shapes(B, LQ, RQ, H + D), shapes(B, LK, RK, H + D), shapes(B, LK, RK, H + D)
    f = lambda x: tpa.tpa(x, k, v, H)
    calls = dict(vmap=lambda: torch.vmap(f)(shapes(3, B, LQ, RQ, H + D)), grad=lambda: torch.func.grad(lambda x: f(x).sum())(q),
                 vjp=lambda: torch.func.vjp(f, q), jvp=lambda: torch.func.jvp(f, (q,), (q,)))
    with pytest.raises(RuntimeError, match="forward-mode|functorch|data pointer"):
        calls[transform]()
