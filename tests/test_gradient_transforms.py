"""The gradient of approx_topk.experimental.differentiable under autograd's transforms.  The native
calls are replaced by plain torch (their results are compared on the GPU in test_gpu_gradient.py); the wrapper,
the operators and the dispatcher are the real ones.  The expectation is the same wrapper with zeros
and a scatter in plain torch for its backward, which every transform has a rule for."""
import pytest
import torch
from torch.autograd import forward_ad

import oracle


@pytest.fixture(autouse=True)
def native_calls_in_plain_torch(monkeypatch):
    from approx_topk import _native

    def two_stage(xs, k0, j, k, layout, index_dtype=torch.int64, want_values=True):
        return oracle.topk(xs.detach(), k, -1, j=j, k_mult=k0 // k, interleaved=layout == _native.INTERLEAVED)

    def stage1(xs, k0, j, layout, index_dtype=torch.int64, want_values=True):
        return two_stage(xs, k0, j, k0, layout)

    def topk_grad(grad_values, indices, n, k0, j, layout):
        # (only ever given plain tensors: what has a derivative or a batch dim is dealt with before)
        assert not torch._C._functorch.is_functorch_wrapped_tensor(grad_values)
        assert not torch._C._functorch.is_functorch_wrapped_tensor(indices)
        out = torch.zeros(indices.shape[:-1] + (n,), dtype=grad_values.dtype)
        return out.scatter_(-1, indices, grad_values.detach())

    monkeypatch.setattr(_native, "require_gpu", lambda xs: None)
    monkeypatch.setattr(_native, "topk", two_stage)
    monkeypatch.setattr(_native, "stage1", stage1)
    monkeypatch.setattr(_native, "topk_grad", topk_grad)


class _Plain(torch.autograd.Function):
    @staticmethod
    def forward(ctx, xs, k, j, k_mult):
        values, indices = oracle.topk(xs, k, -1, j=j, k_mult=k_mult)
        ctx.shape = xs.shape
        ctx.save_for_backward(indices)
        ctx.mark_non_differentiable(indices)
        return values, indices

    @staticmethod
    def backward(ctx, grad_values, _):
        return grad_values.new_zeros(ctx.shape).scatter(-1, ctx.saved_tensors[0], grad_values), None, None, None


def _both(seed=0, j=2, k_mult=2):
    """(values, x, w) of the wrapper and of the plain one."""
    from approx_topk.experimental.differentiable import topk
    out = []
    for kind in range(2):
        x = torch.randn(3, 2, 64, generator=torch.Generator().manual_seed(seed)).requires_grad_()
        values, _ = topk(x, 8, -1, j=j, k_mult=k_mult) if kind == 0 else _Plain.apply(x, 8, j, k_mult)
        out.append((values, x))
    w = torch.randn(out[0][0].shape, generator=torch.Generator().manual_seed(seed + 1))
    return out, w


@pytest.mark.parametrize("k_mult", [1, 2])
def test_forward_mode_over_the_backward(k_mult):
    pairs, w = _both(k_mult=k_mult)
    tangent = torch.randn(w.shape, generator=torch.Generator().manual_seed(9))
    got, by_level = [], []
    for values, x in pairs:
        def backward(g):
            return torch.autograd.grad(values, x, g, retain_graph=True)[0]
        got.append(torch.func.jvp(backward, (w,), (tangent,)))
        with forward_ad.dual_level():
            by_level.append(forward_ad.unpack_dual(backward(forward_ad.make_dual(w, tangent))))
    for pair in (got, by_level):
        for a, b in zip(*pair):
            assert a is not None and torch.equal(a, b)
    assert got[0][1].abs().sum() > 0


def test_forward_mode_of_forward_mode():
    # the gradient is linear in w: so is every derivative along a path through w that is not
    pairs, w = _both()
    tangent = torch.ones_like(w)
    out = []
    for values, x in pairs:
        def backward(g):
            return torch.autograd.grad(values, x, g ** 3, retain_graph=True)[0]
        out.append(torch.func.jvp(lambda g: torch.func.jvp(backward, (g,), (tangent,))[1], (w,), (tangent,)))
    for a, b in zip(*out):
        assert torch.equal(a, b) and a.abs().sum() > 0


def test_batched_cotangents():
    pairs, w = _both()
    batch = torch.randn((5,) + w.shape, generator=torch.Generator().manual_seed(3))
    got = [torch.autograd.grad(values, x, batch, is_grads_batched=True, retain_graph=True)[0] for values, x in pairs]
    assert got[0].shape == (5, 3, 2, 64) and torch.equal(*got)
    # the batch in another dim, nested, and together with forward mode
    last = torch.moveaxis(batch, 0, -1)
    nested = torch.stack([batch, 2 * batch])
    out = []
    for values, x in pairs:
        def backward(g):
            return torch.autograd.grad(values, x, g, retain_graph=True)[0]
        vmap, jvp = torch.func.vmap, torch.func.jvp
        out.append((vmap(backward, in_dims=-1)(last), vmap(backward, in_dims=-1, out_dims=1)(last),
                    vmap(vmap(backward))(nested),
                    vmap(lambda g: jvp(backward, (g,), (g,))[1])(batch),
                    jvp(vmap(backward), (batch,), (batch,))[1]))
    for a, b in zip(*out):
        assert torch.equal(a, b) and a.abs().sum() > 0


def test_batched_cotangents_go_through_one_call(monkeypatch):
    from approx_topk import _native
    calls, inner = [], _native.topk_grad
    monkeypatch.setattr(_native, "topk_grad", lambda *a: (calls.append(a[0].shape), inner(*a))[1])
    ((values, x), _), w = _both()
    torch.func.vmap(lambda g: torch.autograd.grad(values, x, g)[0])(w.expand((7,) + w.shape))
    assert calls == [(7,) + w.shape]


def test_reverse_mode_over_the_backward():
    pairs, w = _both()
    for create in (True, False):
        out = []
        for values, x in pairs:
            g = w.clone().requires_grad_()
            (grad,) = torch.autograd.grad((values ** 2 * g).sum(), x, create_graph=create, retain_graph=True)
            assert grad.requires_grad == create
            if create:
                out.append(torch.autograd.grad((grad ** 2).sum(), (x, g), retain_graph=True))
            else:
                out.append((grad,))
        for a, b in zip(*out):
            assert torch.equal(a, b) and a.abs().sum() > 0


def test_direct_calls_of_the_operator_are_differentiable():
    op = torch.ops.approx_topk.topk_grad.default
    x = torch.randn(3, 64, generator=torch.Generator().manual_seed(1))
    _, indices = oracle.topk(x, 8, -1, j=2)
    w = torch.randn(3, 8, requires_grad=True)
    out = op(w, indices, 64, 8, 2, True)
    g = torch.randn(3, 64)
    (back,) = torch.autograd.grad(out, w, g)
    assert torch.equal(back, g.gather(1, indices))
    with torch.no_grad():
        assert not op(w, indices, 64, 8, 2, True).requires_grad
    with torch.inference_mode():
        assert torch.equal(op(w, indices, 64, 8, 2, True), out)
    # indices with a batch dim of their own
    many = torch.stack([indices, indices.flip(0)])
    got = torch.func.vmap(lambda i: op(w.detach(), i, 64, 8, 2, True))(many)
    assert torch.equal(got, torch.stack([torch.zeros(3, 64).scatter(1, i, w.detach()) for i in many]))
    assert torch.equal(torch.func.jacrev(lambda v: op(v, indices, 64, 8, 2, True))(w.detach()),
                       torch.func.jacfwd(lambda v: op(v, indices, 64, 8, 2, True))(w.detach()))


class _Drops(torch.autograd.Function):
    """Sums its input and hands no gradient back."""
    @staticmethod
    def forward(ctx, values):
        return values.sum()

    @staticmethod
    def backward(ctx, g):
        return None


def test_a_missing_gradient_of_the_values_counts_as_zeros():
    pairs, _ = _both()
    for values, x in pairs:
        (grad,) = torch.autograd.grad(_Drops.apply(values), x)
        assert grad.shape == x.shape and grad.dtype == x.dtype and not grad.any()
    from approx_topk.experimental.differentiable import topk
    for dtype in (torch.float16, torch.float64):
        x = torch.randn(2, 64).to(dtype).requires_grad_()
        _Drops.apply(topk(x, 8, -1)[0]).backward()
        assert x.grad.dtype == dtype and x.grad.shape == x.shape and not x.grad.any()


def _nodes():
    """The wrapper's node in Python and the native one, which it takes for plain GPU tensors."""
    from approx_topk import _native
    from approx_topk.experimental import differentiable
    yield differentiable._TopkWithGradient.apply
    yield _native.host.differentiable_topk


@pytest.mark.parametrize("wrapped", [False, True])
def test_backward_under_compiled_autograd(wrapped):
    # the forward runs eagerly, the backward through a graph that compiled autograd builds of its nodes
    from torch._dynamo import compiled_autograd
    for node in _nodes():
        x = torch.randn(3, 64, generator=torch.Generator().manual_seed(2)).requires_grad_()
        values, indices = node(x * 2 if wrapped else x, 8, -1, 2, 2, True, False)
        assert values.requires_grad and not indices.requires_grad and indices.grad_fn is None
        w = torch.randn(values.shape, generator=torch.Generator().manual_seed(4))
        with compiled_autograd._enable(lambda graph: torch.compile(graph, backend="eager")):
            (values * w).sum().backward()
        want = torch.zeros(3, 64).scatter(-1, indices, w) * (2 if wrapped else 1)
        assert torch.equal(x.grad, want)


def test_function_modes_see_the_gradient_operator():
    from torch.overrides import TorchFunctionMode

    class Seen(TorchFunctionMode):
        def __init__(self):
            super().__init__()
            self.calls = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.calls.append(func)
            return func(*args, **(kwargs or {}))

    for node in _nodes():
        x = torch.randn(3, 64, generator=torch.Generator().manual_seed(2)).requires_grad_()
        values, indices = node(x, 8, -1, 2, 2, True, False)
        with Seen() as mode:
            torch.autograd.backward((values,), (torch.ones(3, 8),))
        assert torch.ops.approx_topk.topk_grad.default in mode.calls
        assert torch.equal(x.grad, torch.zeros(3, 64).scatter(-1, indices, 1.0))
