"""The native host path of the operators (csrc/host_binding.cpp) against the Python functions that take every
other call: the forms it accepts and those it hands on, the errors, and the gradient's node under what
autograd does to it."""
import pytest
import torch
from torch.autograd import forward_ad

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16, torch.float64, torch.uint8, torch.int8, torch.int16,
          torch.int32, torch.int64]


def _general(monkeypatch, call):
    """`call()` with the Python path alone."""
    from approx_topk import _native
    _native.lib()  # (bound once, with the module in place)
    with monkeypatch.context() as m:
        m.setattr(_native, "host", None)
        return call()


def _forms(dtype):
    g = torch.Generator().manual_seed(3)

    def make(*shape):
        return torch.randint(0, 100, shape, generator=g).to(dtype).cuda()

    yield make(512)
    yield make(3, 512)
    yield make(2, 3, 512)
    yield make(3, 1000)[:, 488:]             # rows of a wider matrix
    yield make(3, 1024)[:, ::2]              # no unit stride
    yield make(512, 3).t()
    yield make(6, 4, 512)[::2]
    yield make(3, 1, 512).expand(3, 4, 512)
    yield make(1537)[1:]                     # off 16 bytes
    yield make(0, 512)


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_every_form_as_in_python(dtype, monkeypatch):
    from approx_topk import topk
    from approx_topk.experimental import bucketed_argmax, compact_indices
    from approx_topk.priority_queue import _topk
    for x in _forms(dtype):
        for kw in (dict(), dict(j=2), dict(j=4, k_mult=2), dict(k_mult=4, interleaved=False), dict(j=2, interleaved=False)):
            want = _general(monkeypatch, lambda: _topk(x, 16, -1, **kw))
            for got in (topk(x, 16, -1, **kw), topk(x, 16, x.ndim - 1, **kw), _topk(x, 16, -1, **kw)):
                assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), (x.shape, x.stride(), kw)
                assert got[0].dtype == dtype and got[1].dtype == torch.int64 and got[0].is_contiguous()
            narrow = compact_indices.topk(x, 16, -1, **kw)
            assert narrow[1].dtype == torch.int32 and torch.equal(narrow[1].long(), want[1])
            only = compact_indices.topk_indices(x, 16, -1, **kw)
            assert torch.equal(only.long(), want[1])
        if x.numel():
            for interleaved in (True, False):
                want = _general(monkeypatch, lambda: bucketed_argmax.topk_triton(x, 48, -1, interleaved))
                got = bucketed_argmax.topk_triton(x, 48, -1, interleaved)
                assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_which_calls_the_module_takes():
    from approx_topk import _native
    x = torch.randn(3, 512).cuda()
    _native.lib()
    for t in (x, x[0], x[1:], torch.nn.Parameter(x), x.clone().requires_grad_(), x.view(3, 2, 256)):
        assert _native.host.run(t, 16, 1, 16, _native.INTERLEAVED, False, True, False) is not None
    for t in (x[:, ::2], x.t(), x[:0], x[:, :500], x.cpu(), x.bool(), torch.complex(x, x).conj(), x.to_sparse()):
        assert _native.host.run(t, 16, 1, 16, _native.INTERLEAVED, False, True, False) is None


@pytest.mark.parametrize("args,kwargs", [
    ((0, -1), {}), ((-1, -1), {}), ((4, 0), {}), ((64, 0), dict(j=1)), ((65, -1), {}), ((8, -1), dict(j=3)), ((8, -1), dict(j=5)),
    ((8, -1), dict(j=0)), ((8, -1), dict(k_mult=0)), ((8, -1), dict(k_mult=1 << 62)), ((8, 5), {}), ((8, -3), {}),
])
def test_what_is_refused_stays_refused(args, kwargs, monkeypatch):
    from approx_topk import topk
    from approx_topk.priority_queue import _topk
    x = torch.randn(3, 64).cuda()

    def outcome(fn):
        try:
            values, indices = fn(x, *args, **kwargs)
            return values.shape, indices.shape
        except Exception as e:
            return type(e), str(e).splitlines()[0]

    assert outcome(topk) == _general(monkeypatch, lambda: outcome(_topk))


@pytest.mark.parametrize("args", [(8.0, -1), ("8", -1), (8, -1.0), (1 << 70, -1), (8, -1, 1, 1, "no"), (8, -1, 1, None), (None, -1),
                                  (8, -1, True, True, 1, None), (torch.tensor(8), -1)], ids=str)
def test_arguments_of_other_types_as_in_python(args, monkeypatch):
    from approx_topk.experimental import bucketed_argmax, compact_indices, differentiable
    x = torch.randn(3, 64).cuda()

    def outcome(fn):
        try:
            values, indices = fn()
            return values.cpu().tolist(), indices.cpu().tolist()
        except Exception as e:
            return type(e), str(e).splitlines()[0]

    calls = [lambda: differentiable.topk(x, *args), lambda: compact_indices.topk(x, *args)]
    if len(args) == 2:
        calls.append(lambda: bucketed_argmax.topk_triton(x, *args, True))
    for call in calls:
        assert outcome(call) == _general(monkeypatch, lambda: outcome(call))


def test_other_dtypes_and_devices_are_refused():
    from approx_topk import topk
    with pytest.raises(RuntimeError, match="unsupported dtype"):
        topk(torch.zeros(3, 64, dtype=torch.bool).cuda(), 4, -1)
    with pytest.raises(RuntimeError, match="expected a tensor on a GPU"):
        topk(torch.zeros(3, 64), 4, -1)


def _pair(shape=(3, 5, 256), seed=0, dtype=torch.float64):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=g, dtype=dtype).cuda()


def _expect(x, indices, grad):
    return torch.zeros_like(x).scatter(-1, indices, grad)


@pytest.mark.parametrize("form", ["tensor", "parameter", "columns", "expanded", "hooks", "retained"])
def test_gradient_node(form):
    from approx_topk.experimental.differentiable import topk
    x = _pair()
    leaf = torch.nn.Parameter(x) if form == "parameter" else x.clone().requires_grad_()
    xs = leaf[..., ::2] if form == "columns" else leaf[:1].expand(4, 5, 256) if form == "expanded" else leaf
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t.cpu(), lambda t: t.cuda()) \
            if form == "hooks" else torch.enable_grad():
        values, indices = topk(xs, 16, -1, j=2, k_mult=2)
    assert values.requires_grad and not indices.requires_grad and indices.grad_fn is None
    assert torch.equal(values, xs.gather(-1, indices))
    grad = _pair(values.shape, 1)
    (got,) = torch.autograd.grad(values, leaf, grad, retain_graph=True)
    (want,) = torch.autograd.grad(xs.gather(-1, indices), leaf, grad, retain_graph=True)
    assert torch.equal(got, want) and (len(packed) == 1) == (form == "hooks")
    if form == "retained":
        assert torch.equal(torch.autograd.grad(values, leaf, grad)[0], want)
        with pytest.raises(RuntimeError):
            torch.autograd.grad(values, leaf, grad)


def test_gradient_node_under_transforms():
    from approx_topk.experimental.differentiable import topk
    x = _pair().requires_grad_()
    values, indices = topk(x, 16, -1, j=2, k_mult=2)
    grad = _pair(values.shape, 1).requires_grad_()
    # reverse over reverse: linear in the gradient, and the second derivative of a gather
    (first,) = torch.autograd.grad(values.square().sum() + (values * grad).sum(), x, create_graph=True)
    (second,) = torch.autograd.grad(first.square().sum(), x, retain_graph=True)
    want = _expect(x, indices, (2 * (2 * values + grad)) * 2).detach()
    torch.testing.assert_close(second, want)
    # a batch of gradients, and forward mode through the backward
    batch = torch.stack([grad.detach(), 2 * grad.detach()])
    (many,) = torch.autograd.grad(values, x, batch, is_grads_batched=True, retain_graph=True)
    assert torch.equal(many[1], 2 * many[0]) and torch.equal(many[0], _expect(x, indices, grad).detach())
    with forward_ad.dual_level():
        dual = forward_ad.make_dual(grad.detach(), 3 * grad.detach())
        (out,) = torch.autograd.grad(values, x, dual, retain_graph=True)
        primal, tangent = forward_ad.unpack_dual(out)
        assert torch.equal(primal, many[0]) and torch.equal(tangent, 3 * many[0])
    vjp = torch.func.vmap(lambda g: torch.autograd.grad(values, x, g, retain_graph=True)[0])(batch)
    assert torch.equal(vjp, many)
    # unused values, and a result that is saved and changed
    (none,) = torch.autograd.grad(topk(x, 16, -1)[0].sum() * 0 + x.sum() * 0, x)
    assert not none.any()
    values, indices = topk(x, 16, -1)
    indices.add_(0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(values.sum(), x)
    with torch.no_grad():
        assert not topk(x, 16, -1)[0].requires_grad


def test_function_modes_see_the_operators():
    from torch.overrides import TorchFunctionMode
    from approx_topk.experimental.differentiable import topk

    class Seen(TorchFunctionMode):
        def __init__(self):
            super().__init__()
            self.calls = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.calls.append(func)
            return func(*args, **(kwargs or {}))

    x = _pair().requires_grad_()
    want = topk(x, 16, -1, j=2, k_mult=2)
    for forward_too in (True, False):
        mode = Seen()
        if forward_too:
            with mode:
                values, indices = topk(x, 16, -1, j=2, k_mult=2)
            assert torch.ops.approx_topk.topk.default in mode.calls
            assert torch.equal(values, want[0]) and torch.equal(indices, want[1])
        else:
            values, indices = want
        mode.calls.clear()
        with mode:
            torch.autograd.backward((values,), (torch.ones_like(values),))
        assert torch.ops.approx_topk.topk_grad.default in mode.calls
    assert torch.equal(x.grad, 2 * _expect(x, want[1], torch.ones_like(want[0])).detach())


@pytest.mark.parametrize("node", ["native", "python"])
def test_backward_under_compiled_autograd(node):
    from torch._dynamo import compiled_autograd
    from approx_topk.experimental import differentiable
    x = _pair().requires_grad_()
    if node == "native":
        values, indices = differentiable.topk(x, 16, -1, j=2, k_mult=2)
    else:
        values, indices = differentiable._TopkWithGradient.apply(x, 16, -1, 2, 2, True, False)
    assert not indices.requires_grad and indices.grad_fn is None
    grad = _pair(values.shape, 1)
    with compiled_autograd._enable(lambda graph: torch.compile(graph, backend="eager")):
        (values * grad).sum().backward()
    assert torch.equal(x.grad, _expect(x, indices, grad).detach())


def test_threads_and_streams():
    from concurrent.futures import ThreadPoolExecutor
    from approx_topk import topk
    from approx_topk.experimental import differentiable
    want = topk(_pair((64, 4096), dtype=torch.float32), 64, -1, j=2, k_mult=2)
    torch.cuda.synchronize()

    def work(seed):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(50):
                x = _pair((64, 4096), dtype=torch.float32).requires_grad_()
                values, indices = differentiable.topk(x, 64, -1, j=2, k_mult=2)
                (g,) = torch.autograd.grad(values.sum(), x)
                assert torch.equal(values, want[0]) and torch.equal(indices, want[1]) and int(g.sum()) == 64 * 64
        return seed

    with ThreadPoolExecutor(4) as pool:  # (result() raises what a worker raised)
        assert [f.result(timeout=100) for f in [pool.submit(work, s) for s in range(4)]] == [0, 1, 2, 3]
