"""Products of split operands (``csrc/split_bf16.hpp``) at the ends of float32's range: operands down to the
smallest subnormal against large partners, through every kernel that splits, against float64 of the same
inputs.

Tolerance: as for ordinary operands, 4e-7 + 3e-8 K of the sum of |a b| (see ``test_gates_gpu.py``); the
products are ordinary numbers, so no result is subnormal."""
import pytest
import torch

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from ictc_o3.backends.hip import degree_linear as D  # noqa: E402
from ictc_o3.backends.hip import gates as G  # noqa: E402

DEV = torch.device("cuda", 0)


def _at(exponent, *shape):
    """Values of random sign whose magnitudes lie in [2^exponent, 2^(exponent + 1)), rounded to float32 (to its
    subnormals where the exponent is below -126)."""
    gen = torch.Generator().manual_seed(-exponent)
    v = (1 + torch.rand(*shape, generator=gen, dtype=torch.float64)) * 2.0 ** exponent
    return (v * (torch.randint(0, 2, shape, generator=gen) * 2 - 1)).float().to(DEV)


def _partner(exponent):
    """Exponent of partners whose products with 2^exponent are ordinary (below 2^103, where the kernels turn
    to plain float32)."""
    return min(-exponent - 5, 100)


def _close(got, a, b):
    a, b = a.double(), b.double()
    assert bool(torch.isfinite(got).all())
    over = ((got.double() - a @ b).abs() / (a.abs() @ b.abs())).max()
    assert over <= 4e-7 + 3e-8 * a.shape[1], f"{over:.2e} of the sum of |a b|"


@pytest.mark.parametrize("small", [-104, -112, -116, -120, -124, -126, -130, -140, -149])
def test_gates_products_of_small_operands(small):
    edges, width, large = 200, 68, _partner(small)
    for eh, ew, eg in ((small, large, large), (large, small, small)):
        h, w, g = _at(eh, edges, 64), _at(ew, width, 64), _at(eg, edges, width)
        _close(G._forward(h, w, None), h, w.t())
        _close(G._weight_grad(g, h, False), g.t(), h)
        w = _at(_partner(eg), width, 64)
        _close(G._input_grad(g, w, None), g, w)


@pytest.mark.parametrize("small", [-112, -118, -126, -140, -149])
def test_linear_products_of_small_operands(small):
    plan = D.DegreeLinearPlan((2, 1), 64, 64)
    nodes, large = 5000, _partner(small)                   # a block for every CU: the split kernels
    for ex, ew in ((small, large), (large, small)):
        x, gy = _at(ex, nodes, plan.in_width), _at(ex, nodes, plan.out_width)
        ws = [_at(ew, 64, 64 * k) for k in (2, 1)]
        y, gx = D._forward_raw(plan, x, ws, 1.0), D._input_grad_raw(plan, gy, ws, 1.0)
        gy2 = _at(_partner(ex), nodes, plan.out_width)
        gw = D._weight_grad_raw(plan, 0, gy2, x, 1.0, [True, True])
        for l in range(2):
            _close(plan.y_rows(y, l), plan.x_rows(x, l), ws[l].t())
            _close(plan.x_rows(gx, l), plan.y_rows(gy, l), ws[l])
            _close(gw[l], plan.y_rows(gy2, l).t(), plan.x_rows(x, l))
