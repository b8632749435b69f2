"""The C++ autograd kernels of the torch operators, on a trilinear product defined for the CPU through the same registration
as the operators: derivatives of three orders, graphs that are not asked for, and the transforms of torch around them."""
import contextlib

import pytest
import torch

from openequivariance_amd.autograd_glue import define_derivatives, define_operator, double_backward_terms

OPERANDS, INDEX = ("x", "y", "w"), ("rows", "cols")


def like(*tensors):
    return [t.new_empty(*t.shape) for t in tensors]


@pytest.fixture(scope="module")
def ops():
    calls = []

    def forward_impl(x, y, w, rows, cols):
        calls.append("forward")
        return torch.zeros_like(x).index_add_(0, rows, (x[cols] * y * w))

    def backward_impl(x, y, w, g, rows, cols):
        calls.append("backward")
        g = g[rows]
        return [torch.zeros_like(x).index_add_(0, cols, g * y * w), g * x[cols] * w, g * x[cols] * y]

    forward = define_operator("glue_forward", OPERANDS + INDEX, "Tensor", forward_impl, lambda x, *rest: like(x)[0], "CPU")
    backward = define_operator("glue_backward", (*OPERANDS, "L3_grad", *INDEX), "Tensor[]", backward_impl,
                               lambda x, y, w, *rest: like(x, y, w), "CPU")
    define_derivatives("glue_forward", "glue_backward", OPERANDS + INDEX,
                       lambda x, y, w, g, a, b, v, *index: list(double_backward_terms(forward, backward, x, y, w, g, a, b, v, index)))
    return forward, backward, calls


@pytest.fixture
def data():
    gen = torch.Generator().manual_seed(3)
    x, y, w = (torch.randn(n, 4, generator=gen, dtype=torch.float64, requires_grad=True) for n in (5, 9, 9))
    return (x, y, w), (torch.randint(0, 5, (9,), generator=gen), torch.randint(0, 5, (9,), generator=gen))


def reference(x, y, w, rows, cols):
    return torch.zeros_like(x).index_add(0, rows, x[cols] * y * w)


def test_derivatives_of_three_orders(ops, data):
    (args, index), got = data, []
    for f in (ops[0], reference):
        z = f(*args, *index)
        first = torch.autograd.grad(z.square().sum(), args, create_graph=True)
        second = torch.autograd.grad(first[0].square().sum() + first[2].sin().sum(), args, create_graph=True)   # no cotangent of dy
        third = torch.autograd.grad(sum(t.cos().sum() for t in second), args)
        got.append((z, *first, *second, *third))
    for a, b in zip(*got):
        assert torch.allclose(a, b, rtol=1e-12, atol=1e-12)
    assert torch.autograd.gradgradcheck(lambda *a: ops[0](*a, *index), args)


def test_graph_only_where_one_is_asked_for(ops, data):
    (x, y, w), index = data
    with torch.no_grad():
        assert not ops[0](x, y, w, *index).requires_grad
    plain = [t.detach() for t in (x, y, w)]
    assert not ops[0](*plain, *index).requires_grad
    g, = torch.autograd.grad(ops[0](plain[0], y, plain[2], *index).sum(), y)          # one of the operands
    assert torch.allclose(g, torch.autograd.grad(reference(plain[0], y, plain[2], *index).sum(), y)[0])
    del ops[2][:]
    z = ops[0](x, y, w, *index)
    first = torch.autograd.grad(z.sum(), (x, y, w))
    assert ops[2] == ["forward", "backward"] and not any(t.requires_grad for t in first)
    z = ops[0](x, y, w, *index)                          # the caller's operands may change between the passes, as before
    with torch.no_grad():
        x.mul_(2)
    torch.autograd.grad(z.sum(), (x, y, w))
    z = ops[0](x, y, w, *index)                          # and the pass back may be taken twice
    a, b = (torch.autograd.grad(z.sum(), w)[0] for _ in range(2))
    assert torch.equal(a, b)


def test_transforms(ops, data):
    (x, y, w), index = data
    want = torch.autograd.grad(reference(x, y, w, *index).sin().sum(), (x, y, w))
    run = lambda a: ops[0](a, y, w, *index).sin()
    z = torch.utils.checkpoint.checkpoint(run, x, use_reentrant=False)
    assert torch.allclose(torch.autograd.grad(z.sum(), x)[0], want[0])
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        assert torch.allclose(torch.autograd.grad(run(x).sum(), x)[0], want[0])
    compiled = torch.compile(lambda *a: ops[0](*a, *index).sin().sum(), backend="aot_eager", fullgraph=True)
    for a, b in zip(torch.autograd.grad(compiled(x, y, w), (x, y, w)), want):
        assert torch.allclose(a, b)
    plain = [t.detach() for t in (x, y, w)]
    many = torch.func.vmap(lambda a: ops[0](a, *plain[1:], *index))(torch.stack([plain[0], 2 * plain[0]]))
    assert torch.allclose(many[1], 2 * reference(*plain, *index))
    torch.library.opcheck(ops[0], (x, y, w, *index), test_utils=("test_schema", "test_faketensor", "test_autograd_registration"))
    torch.library.opcheck(ops[1], (x, y, w, x.detach(), *index), test_utils=("test_schema", "test_faketensor", "test_autograd_registration"))


def test_compiled_autograd(ops, data):
    """Backward passes as torch records and compiles them, of two operators whose nodes differ only in their rule."""
    (args, index), compiler = data, torch.compile(backend="aot_eager")
    negative = define_operator("glue_negative", OPERANDS + INDEX, "Tensor", lambda *a: -2 * ops[0](*a), lambda x, *rest: like(x)[0], "CPU")
    negative_backward = define_operator("glue_negative_backward", (*OPERANDS, "L3_grad", *INDEX), "Tensor[]",
                                        lambda *a: [-2 * t for t in ops[1](*a)], lambda x, y, w, *rest: like(x, y, w), "CPU")
    define_derivatives("glue_negative", "glue_negative_backward", OPERANDS + INDEX,
                       lambda x, y, w, g, a, b, v, *index: list(double_backward_terms(negative, negative_backward, x, y, w, g, a, b, v, index)))
    import torch._dynamo.compiled_autograd as compiled_autograd

    def gradients(f, around):
        first, got = torch.autograd.grad(f(*args, *index).sin().sum(), args, create_graph=True), []
        for loss in (f(*args, *index).sin().sum(), sum(t.square().sum() for t in first)):      # both kinds of node
            with around():
                loss.backward()
            got += [t.grad for t in args]
            for t in args:
                t.grad = None
        return got

    for op, scale in ((ops[0], 1), (negative, -2)) * 2:
        got = gradients(op, lambda: compiled_autograd._enable(compiler))
        want = gradients(lambda *a: scale * reference(*a), contextlib.nullcontext)
        assert all(torch.allclose(a, b, rtol=1e-12, atol=1e-12) for a, b in zip(got, want))
