"""The kernel behind the gradient of approx_topk.experimental.differentiable against zeros and a
scatter in plain torch: bits are moved to distinct positions, so the two are equal."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (rows, n, k, j, k_mult): rows of one tile and of one element more; few entries over many tiles;
# column tiles with every sub-row and with runs of them, all of a bucket's entries kept and
# found by search; the last column tile, sub-row and run not full
SHAPES = [
    (3, 64, 16, 4, 1),
    (3, 16384, 4096, 2, 1), (2, 16385, 4096, 2, 1), (2, 32769, 2048, 1, 4),
    (2, 400003, 60, 2, 2), (3, 100003, 1024, 1, 1),
    (2, 1 << 18, 16384, 2, 1), (2, 300007, 18750, 2, 1), (2, 300007, 4690, 2, 4),
    (1, 1 << 20, 2048, 1, 1), (1, (1 << 21) + 77, 1540, 4, 1), (1, (1 << 21) + 77, 1540, 4, 2),
    (1, 1 << 19, 2052, 2, 1),
]


@pytest.mark.parametrize("interleaved", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16, torch.float64],
                         ids=lambda d: str(d).split(".")[-1])
def test_gradient_kernel_equals_a_scatter(dtype, interleaved):
    from approx_topk.experimental.differentiable import topk
    for rows, n, k, j, k_mult in SHAPES:
        g = torch.Generator(device="cuda").manual_seed(n + k)
        x = torch.randn(rows, n, generator=g, device="cuda").to(dtype).requires_grad_()
        values, indices = topk(x, k, -1, j=j, k_mult=k_mult, interleaved=interleaved)
        w = torch.randn(rows, k, generator=g, device="cuda").to(dtype)
        (grad,) = torch.autograd.grad(values, x, w)
        expect = torch.zeros_like(x).scatter(1, indices, w)
        assert torch.equal(grad, expect), (rows, n, k, j, k_mult)


# batches whose tiles hold several rows: two of them and a last tile of one; as many as a tile has room for, and
# a last tile of fewer; rows of one element; two rows to a tile of 64 KiB in four-byte types, then only one
SHORT = [
    (1025, 7, 3, 1, 1), (5003, 64, 16, 4, 1), (40003, 1001, 20, 2, 2), (2049, 1, 1, 1, 1),
    (2101, 8192, 60, 2, 2), (2101, 8193, 60, 2, 2), (1024, 64, 16, 4, 2),
]


@pytest.mark.parametrize("interleaved", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.float64], ids=lambda d: str(d).split(".")[-1])
def test_short_rows_share_a_tile(dtype, interleaved):
    from approx_topk.experimental.differentiable import topk
    for rows, n, k, j, k_mult in SHORT:
        g = torch.Generator(device="cuda").manual_seed(n + k)
        x = torch.randn(rows, n, generator=g, device="cuda").to(dtype).requires_grad_()
        values, indices = topk(x, k, -1, j=j, k_mult=k_mult, interleaved=interleaved)
        w = torch.randn(rows, k, generator=g, device="cuda").to(dtype)
        (grad,) = torch.autograd.grad(values, x, w)
        assert torch.equal(grad, torch.zeros_like(x).scatter(1, indices, w)), (rows, n, k, j, k_mult)


def test_gradient_of_sums_of_views_and_of_unused_values():
    from approx_topk.experimental.differentiable import topk
    x = torch.randn(2, 3, 5000, device="cuda", requires_grad=True)
    values, indices = topk(x, 40, -1, j=2, k_mult=2)
    (grad,) = torch.autograd.grad(values.sum(), x)   # an expanded gradient
    assert torch.equal(grad, torch.zeros_like(x).scatter(2, indices, 1.0))
    values, _ = topk(x, 40, -1)
    assert torch.equal(torch.autograd.grad(x.sum() + 0 * values.sum(), x)[0], torch.ones_like(x))
    topk(x, 40, -1)   # nothing of it used
    assert torch.equal(torch.autograd.grad(x.sum(), x)[0], torch.ones_like(x))


def test_gradient_of_the_gradient():
    from approx_topk.experimental.differentiable import topk
    x = torch.randn(2, 4096, device="cuda", requires_grad=True)
    values, _ = topk(x, 64, -1, j=2)
    (grad,) = torch.autograd.grad((values ** 3).sum(), x, create_graph=True)
    (second,) = torch.autograd.grad(grad.sum(), x)
    _, indices = topk(x.detach(), 64, -1, j=2)
    expect = torch.zeros_like(x).scatter(1, indices, 6 * x.detach().gather(1, indices))
    assert torch.allclose(second, expect, rtol=1e-6, atol=0)   # one rounding of a product each


def test_transforms_of_the_backward():
    # forward mode of both kinds, batches and both together, next to zeros and a scatter (autograd runs the
    # backward in a thread of its own on a GPU)
    from torch.autograd import forward_ad
    from approx_topk.experimental.differentiable import topk
    x = torch.randn(3, 5000, device="cuda", requires_grad=True)
    values, indices = topk(x, 40, -1, j=2, k_mult=2)
    w, t = torch.randn(2, 3, 40, device="cuda")
    many = torch.randn(5, 3, 40, device="cuda")

    def backward(g):
        return torch.autograd.grad(values, x, g, retain_graph=True)[0]

    def expect(g):
        return g.new_zeros(g.shape[:-1] + (5000,)).scatter(-1, indices.expand(g.shape), g)

    primal, tangent = torch.func.jvp(backward, (w,), (t,))
    assert torch.equal(primal, expect(w)) and torch.equal(tangent, expect(t))
    with forward_ad.dual_level():
        primal, tangent = forward_ad.unpack_dual(backward(forward_ad.make_dual(w, t)))
        assert torch.equal(primal, expect(w)) and torch.equal(tangent, expect(t))
    assert torch.equal(torch.autograd.grad(values, x, many, is_grads_batched=True, retain_graph=True)[0], expect(many))
    assert torch.equal(torch.func.vmap(backward)(many), expect(many))
    assert torch.equal(torch.func.vmap(lambda g: torch.func.jvp(backward, (g,), (g,))[1])(many), expect(many))
    assert torch.equal(torch.func.jvp(torch.func.vmap(backward), (many,), (many,))[1], expect(many))


def test_gradient_operator_under_compile():
    from approx_topk.experimental.differentiable import topk
    x = torch.randn(3, 4096, device="cuda")
    _, indices = topk(x, 64, -1, j=2)
    w = torch.randn(3, 64, device="cuda")
    op = torch.ops.approx_topk.topk_grad.default
    torch.library.opcheck(op, (w, indices, 4096, 64, 2, True),
                          test_utils=("test_schema", "test_faketensor"))

    # a function compiled whole, its backward through the operator
    def loss(x, w):
        values, _ = topk(2 * x, 64, -1, j=2, k_mult=2)
        return (values * w).sum()

    x.requires_grad_()
    (eager,) = torch.autograd.grad(loss(x, w), x)
    graphs = []

    def backend(graph, example_inputs):
        graphs.append(graph.print_readable(print_output=False))
        return make_boxed_func(graph)

    from functorch.compile import make_boxed_func
    from torch._dynamo.backends.common import aot_autograd
    compiled = torch.compile(loss, fullgraph=True, backend=aot_autograd(fw_compiler=backend, bw_compiler=backend))
    (grad,) = torch.autograd.grad(compiled(x, w), x)
    assert torch.equal(grad, eager) and len(graphs) == 2 and "approx_topk.topk_grad" in graphs[1], graphs
