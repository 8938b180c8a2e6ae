"""What the tensor product's path weight must be for the kernels to fold it into the gates
(``gates_and_weight``): every other weight takes the separate product ``gates * weight``, as before the
kernels took one.  CPU only (no kernel runs)."""
import copy

import pytest
import torch

from ictc_o3.backends.hip import tensor_product as T
from ictc_o3.basis.ictd_irreps import EdgeWeightedPathPreservingTensorProduct

ROWS, C = 3, 4


def _owner(lmax=2):
    owner = EdgeWeightedPathPreservingTensorProduct(C, lmax, internal_compute_dtype=torch.float32)
    owner.weight.requires_grad_(False)
    plan = owner.hip_plan(lmax, lmax)
    assert plan.is_full and plan.weight_capacity >= owner.num_paths * C
    return owner, plan, torch.randn(ROWS, owner.num_paths * C)


@pytest.mark.parametrize("shape", [(1, C), (None, 1), (1, 1), (C,), (1, None, C)])
def test_broadcast_weights_take_the_separate_product(shape):
    """The kernels read P * C floats: a weight that broadcasts against [P, C] holds fewer."""
    owner, plan, gates = _owner()
    shape = tuple(owner.num_paths if n is None else n for n in shape)
    owner.weight = torch.nn.Parameter(torch.randn(shape), requires_grad=False)
    product, weight = T.gates_and_weight(owner, plan, gates, ROWS)
    assert weight is None
    want = gates.reshape(ROWS, owner.num_paths, C) * owner.weight
    assert torch.equal(product, want.reshape(ROWS, -1))


def test_a_passed_weight_is_checked():
    owner, plan, gates = _owner()
    x, y = torch.randn(ROWS, 9 * C), torch.randn(ROWS, 9)
    n = owner.num_paths * C
    for bad in (torch.ones(n - 1), torch.ones(owner.num_paths, C), torch.ones(n, dtype=torch.float64),
                torch.ones(2 * n)[::2], torch.ones(n, device="meta"), torch.ones(n, requires_grad=True)):
        with pytest.raises(ValueError):
            T.packed_tensor_product(plan, x, y, gates, bad)
    some = T.TensorProductPlan(owner.paths[1:], C, 2, 2, 2)        # a path subset does not take one
    with pytest.raises(ValueError):
        T.packed_tensor_product(some, x, y, gates[:, C:], torch.ones(n - C))


@pytest.mark.parametrize("change", [lambda w: w.data.mul_(3.0), lambda w: w.mul_(3.0)], ids=["data", "in place"])
def test_the_backward_uses_the_weight_of_its_forward(monkeypatch, change):
    """A weight that changes between a forward and its backward, where only the features are
    differentiated: the gradient is that of the product that was computed."""
    owner, plan, gates = _owner()
    seen = []

    def kernels(plan, x, y, g, w=None, copy=None):
        seen.append(w)
        if copy is not None:
            copy.copy_(w)
        return x.new_zeros(ROWS, plan.full_out_width)

    def adjoint(plan, need, x, y, g, go, w=None):
        seen.append(w.clone())
        return torch.zeros_like(x), None, None

    monkeypatch.setattr(T, "_forward_raw", kernels)
    monkeypatch.setattr(T, "_backward_raw", adjoint)
    x, y = torch.randn(ROWS, 9 * C), torch.randn(ROWS, 9)
    before = owner.weight.reshape(-1).clone()
    out = T.packed_tensor_product(plan, x.requires_grad_(), y, *T.gates_and_weight(owner, plan, gates, ROWS))
    change(owner.weight)
    out.sum().backward()
    assert len(seen) == 2 and torch.equal(seen[1], before)
    # nothing to differentiate: no copy
    T.packed_tensor_product(plan, x.detach(), y, *T.gates_and_weight(owner, plan, gates, ROWS))
    assert seen[2].data_ptr() == owner.weight.data_ptr()


def test_a_forward_mode_tangent_is_not_dropped(monkeypatch):
    """The product has no forward-mode derivative: a weight with a tangent has to reach it with its
    tangent, so that the call is refused and not answered as if there were none."""
    import torch.autograd.forward_ad as fwad
    owner, plan, gates = _owner()
    monkeypatch.setattr(T, "_forward_raw", lambda plan, x, y, g, w=None, copy=None: x.new_zeros(ROWS, plan.full_out_width))
    with fwad.dual_level():
        del owner.weight
        owner.weight = fwad.make_dual(torch.ones(owner.num_paths, C), torch.ones(owner.num_paths, C))
        weight = T.gates_and_weight(owner, plan, gates, ROWS)[1]
        assert fwad.unpack_dual(weight).tangent is not None
        x, y = torch.randn(ROWS, 9 * C), torch.randn(ROWS, 9)
        with pytest.raises(RuntimeError, match="jvp"):
            T.packed_tensor_product(plan, x, y, gates, weight)


def test_a_plan_saved_without_a_weight_capacity():
    """Modules saved whole before plans had the attribute hold plans without it."""
    _, plan, _ = _owner()
    want, saved = plan.weight_capacity, copy.copy(plan)
    saved.__dict__ = {k: v for k, v in plan.__dict__.items() if "capacity" not in k}
    assert saved.weight_capacity == want > 0
