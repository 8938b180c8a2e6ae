"""The TP's frozen path weight folded into the gates by the kernels: bit-identical to multiplying it
into the gates beforehand (values and gradients), for every launch variant and at the rule's edges; live weights, weights too wide for the kernels, path subsets and the
run-time-table degree sets keep the separate product."""
import pytest
import torch

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from ictc_o3 import EdgeTensorProduct  # noqa: E402
from ictc_o3.backends.hip import tensor_product as T  # noqa: E402

DEV = torch.device("cuda", 0)


def _op(channels, lin, le, lout, layout="ir_mul"):
    op = EdgeTensorProduct.create(channels=channels, input_lmax=lin, edge_lmax=le, output_lmax=lout, layout=layout,
                                  device=DEV)
    gen = torch.Generator().manual_seed(channels)
    with torch.no_grad():
        op.tp.weight.copy_(torch.randn(op.tp.num_paths, channels, generator=gen))
    return op


def _inputs(op, rows):
    gen = torch.Generator().manual_seed(rows)
    c = op.tp.channels
    return [torch.randn(rows, w, generator=gen).to(DEV).requires_grad_()
            for w in (c * (op.input_lmax + 1) ** 2, (op.edge_lmax + 1) ** 2, op.gate_width)]


def _everything(call, x, y, g, go, h):
    out = call(x, y, g)
    grads = torch.autograd.grad(out, (x, y, g), go, create_graph=True)
    second = torch.autograd.grad(sum((a * b).sum() for a, b in zip(grads, h)), (x, y, g))
    return [out, *grads, *second]


@pytest.mark.parametrize("channels,lin,le,lout,rows", [(1, 0, 0, 0, 1), (5, 1, 2, 3, 7), (64, 2, 2, 2, 130),
                                                       (128, 3, 3, 3, 33), (192, 2, 1, 2, 9), (24, 3, 2, 1, 64),
                                                       (64, 4, 4, 4, 11), (178, 3, 3, 3, 6), (97, 4, 4, 4, 5)])
def test_folded_weight_equals_the_separate_product(channels, lin, le, lout, rows):
    op = _op(channels, lin, le, lout)
    x, y, g = _inputs(op, rows)
    gates, weight = T.gates_and_weight(op.tp, op.plan, g, rows)
    assert weight is not None and gates.data_ptr() == g.data_ptr()
    go = torch.randn(rows, op.output_width, device=DEV)
    h = [torch.randn_like(t) for t in (x, y, g)]
    plain = lambda a, b, c: T.packed_tensor_product(op.plan, a, b, op.tp.effective_gates(c, rows))   # noqa: E731
    pairs = list(zip(_everything(op, x, y, g, go, h), _everything(plain, x, y, g, go, h)))
    for got, want in pairs[:4]:
        assert torch.equal(got, want)
    # A second derivative is a sum of two substituted maps; the gates' one distributes w over it
    # (w a + w b for w (a + b)): three roundings of 2^-24 for two, at the size of the terms, which
    # N(0, 1) inputs keep within a few times the largest sum.
    for got, want in pairs[4:]:
        assert (got - want).abs().max() <= 16 * 2.0 ** -24 * want.abs().max()


def test_weight_changes_are_seen_and_gates_of_rank_three():
    op = _op(48, 2, 2, 2)
    x, y, g = _inputs(op, 20)
    for change in (lambda w: w.mul_(2.0), lambda w: w.zero_()):
        change(op.tp.weight.data)
        want = T.packed_tensor_product(op.plan, x, y, op.tp.effective_gates(g, 20))
        assert torch.equal(op(x, y, g.reshape(20, op.tp.num_paths, 48)), want)


@pytest.mark.parametrize("channels,degree,rows", [(1, 0, 1), (24, 1, 40), (128, 3, 33), (97, 4, 5)])
def test_the_backward_uses_the_weight_of_its_forward(channels, degree, rows):
    """The kernel's copy of the weight: gradients as before for a weight that changes after the forward."""
    op = _op(channels, degree, degree, degree)
    inputs = _inputs(op, rows)
    go = torch.randn(rows, op.output_width, device=DEV)
    want = torch.autograd.grad(op(*inputs), inputs, go)
    out = op(*inputs)
    op.tp.weight.data.mul_(3.0)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(out, inputs, go), want))


def test_separate_product_where_the_kernels_do_not_take_the_weight():
    op = _op(64, 2, 2, 2)
    x, y, g = _inputs(op, 10)
    op.tp.weight.requires_grad_(True)                       # a live weight: its gradient needs the product
    assert T.gates_and_weight(op.tp, op.plan, g, 10)[1] is None
    out = op(x, y, g)
    gw, = torch.autograd.grad(out.sum(), op.tp.weight)
    assert gw.abs().sum() > 0
    with torch.no_grad():                                   # nothing recorded: folded
        assert T.gates_and_weight(op.tp, op.plan, g, 10)[1] is not None
        assert torch.equal(op(x, y, g), out)
    for args in ((179, 3, 3, 3), (64, 4, 4, 3)):            # P * C above the capacity; run-time path tables
        wide = _op(*args)
        a, b, c = _inputs(wide, 6)
        assert T.gates_and_weight(wide.tp, wide.plan, c, 6)[1] is None
        want = T.packed_tensor_product(wide.plan, a, b, wide.tp.effective_gates(c, 6))
        assert torch.equal(wide(a, b, c), want)
        with pytest.raises(RuntimeError):
            T._forward_raw(wide.plan, a, b, c, wide.tp.weight.reshape(-1))
