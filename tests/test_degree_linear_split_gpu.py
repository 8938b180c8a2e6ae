"""The per-degree linear's split-bf16 kernels at sizes that take them (a block for every CU) and on both sides
of the dispatch's lines: forward, input adjoint, mul_ir maps and weight adjoint against float64, with rows that do not fill a tile, column
chunks that cross a path block (C = 96), a degree without path blocks, outputs wider than a tile, and
non-finite values as in float32.

Tolerance: a product of split operands drops terms below 2^-23 |a b| and every 16 reduction steps round an
fp32 sum at most six times, so an entry of K steps is within about (2^-23 + 6 K / 16 * 2^-24) of the sum of
|a b|; 4e-7 + 3e-8 K of that sum bounds both with room."""
import pytest
import torch

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from ictc_o3.backends.hip import degree_linear as D  # noqa: E402

DEV = torch.device("cuda", 0)
CASES = [((4, 6, 7, 6), 128, 128, 1021), ((1, 2), 96, 96, 5001), ((3, 0, 2), 64, 64, 2503), ((2, 3, 1), 32, 160, 2050),
         ((2, 1), 64, 96, 4100), ((1,), 64, 64, 20003),
         # beside the lines of the dispatch: a single degree's blocks, K of a 64-column tile
         ((4,), 64, 64, 20480), ((4,), 64, 64, 20416), ((1,), 128, 128, 49217), ((1,), 128, 128, 49152),
         ((1, 1, 2), 64, 64, 2100), ((2, 1, 1), 64, 64, 2100),
         ((1, 1, 1, 1), 128, 128, 1024), ((1, 1, 1), 96, 96, 2048), ((1, 1, 1, 1), 96, 96, 2048)]


def _data(counts, c, o, nodes):
    gen = torch.Generator().manual_seed(nodes)
    plan = D.DegreeLinearPlan(counts, c, o)
    x = torch.randn(nodes, plan.in_width, generator=gen).to(DEV)
    gy = torch.randn(nodes, plan.out_width, generator=gen).to(DEV)
    ws = [(torch.randn(o, k * c, generator=gen) / max(1, k * c) ** 0.5).to(DEV) for k in counts]
    return plan, x, gy, ws


def _within(got, a, b):
    over = ((got.double() - a.double() @ b.double()).abs()
            - (4e-7 + 3e-8 * a.shape[1]) * (a.double().abs() @ b.double().abs())).max()
    assert over <= 0, f"{over:.2e} over the bound"


@pytest.mark.parametrize("counts,c,o,nodes", CASES)
def test_products_match_float64(counts, c, o, nodes):
    plan, x, gy, ws = _data(counts, c, o, nodes)
    y, gx = D._forward_raw(plan, x, ws, 1.0), D._input_grad_raw(plan, gy, ws, 1.0)
    gw = D._weight_grad_raw(plan, 0, gy, x, 1.0, [True] * len(counts))
    for l, k in enumerate(counts):
        if k == 0:
            assert not plan.y_rows(y, l).any() and gw[l] is None
            continue
        _within(plan.y_rows(y, l), plan.x_rows(x, l), ws[l].t())
        _within(plan.x_rows(gx, l), plan.y_rows(gy, l), ws[l])
        _within(gw[l], plan.y_rows(gy, l).t(), plan.x_rows(x, l))
    assert torch.equal(D._forward_raw(plan, x, ws, 0.5), 0.5 * y)     # alpha a power of two: exact
    assert torch.equal(D._input_grad_raw(plan, gy, ws, 0.5), 0.5 * gx)


@pytest.mark.parametrize("c,o,lmax,nodes", [(128, 128, 3, 1100), (96, 64, 2, 2100), (64, 128, 1, 4200), (32, 32, 3, 1500),
                                              (128, 64, 2, 2100)])
def test_mul_ir_maps_match_float64(c, o, lmax, nodes):
    plan, _, gy, ws = _data((1,) * (lmax + 1), c, o, nodes)
    x = torch.randn(nodes, c * (lmax + 1) ** 2, device=DEV)
    y = D.degree_linear_mul_ir(x, ws, plan, 1.0)
    gx, *gw = torch.autograd.grad(D.degree_linear_mul_ir(x.requires_grad_(), [w.requires_grad_() for w in ws], plan, 1.0),
                                  (x, *ws), gy)
    back = plan.transposed()
    for l, w in enumerate(ws):
        _within(plan.y_rows(y, l), plan.mul_ir_rows(x, l).detach(), w.detach().t())
        _within(back.y_rows(gx, l), plan.y_rows(gy, l), w.detach())
        _within(gw[l], plan.y_rows(gy, l).t(), plan.mul_ir_rows(x, l).detach())


def test_non_finite_values_as_in_float32():
    plan, x, gy, ws = _data((2, 1), 128, 128, 5000)
    x[7, 3], x[9, 200], x[11, 5] = float("inf"), 3.3999e38, float("nan")
    gy[8, 3], gy[20, 130] = float("-inf"), float("nan")
    y, gx = D._forward_raw(plan, x, ws, 1.0), D._input_grad_raw(plan, gy, ws, 1.0)
    gw = D._weight_grad_raw(plan, 0, gy, x, 1.0, [True, True])
    for l in range(2):
        for got, a, b in ((plan.y_rows(y, l), plan.x_rows(x, l), ws[l].t()),
                          (plan.x_rows(gx, l), plan.y_rows(gy, l), ws[l]),
                          (gw[l], plan.y_rows(gy, l).t(), plan.x_rows(x, l))):
            want = a @ b
            assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
            keep = torch.isfinite(want)
            size = (a.double().abs() @ b.double().abs())[keep]
            assert bool(((got[keep].double() - want[keep].double()).abs() <= 1e-5 * size + 1e-6).all())
