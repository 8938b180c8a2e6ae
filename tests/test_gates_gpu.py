"""The 64-wide edge products (``ictc_hip_gates_*``): gates, input adjoint and weight adjoint against
float64 at the edges of their tiles, in every storage order they accept, with non-finite values, and
the routing rule of ``backends.hip.gates.product``.

Tolerance: a product of split operands drops terms below 2^-23 |a b| and every 16 reduction steps
round an fp32 sum six times, so an entry of K steps is within about (2^-23 + 6 K / 16 * 2^-24) of the
sum of |a b| (worst case); 4e-7 + 3e-8 K of that sum bounds both with room."""
import pytest
import torch

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from ictc_o3.backends.hip import gates as G  # noqa: E402
from ictc_o3.backends.hip import linear as L  # noqa: E402

DEV = torch.device("cuda", 0)


def _inputs(edges, width):
    gen = torch.Generator().manual_seed(1000 * edges + width)
    h, w, g = (torch.randn(*s, generator=gen).to(DEV) for s in ((edges, 64), (width, 64), (edges, width)))
    return h, w / 8, g


def _close(got, a, b):
    expect, bound = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    over = ((got.double() - expect).abs() - (4e-7 + 3e-8 * a.shape[1]) * bound).max()
    assert over <= 0, f"{over:.2e} over the bound"


@pytest.mark.parametrize("edges,width", [(1, 4), (31, 60), (33, 64), (128, 68), (129, 100), (257, 132), (1000, 352),
                                         (4099, 2944)])
def test_products_match_float64(edges, width):
    h, w, g = _inputs(edges, width)
    _close(G._forward(h, w, None), h, w.t())
    _close(G._input_grad(g, w, None), g, w)
    _close(G._weight_grad(g, h, False), g.t(), h)


@pytest.mark.parametrize("edges,width", [(130, 96), (515, 204)])
def test_storage_orders_are_bit_identical(edges, width):
    """A transposed weight, row slices of wider tensors, an output row slice, an odd output row
    stride and the transposed weight gradient."""
    h, w, g = _inputs(edges, width)
    wt = w.t().contiguous().t()
    out, gh, gw = G._forward(h, w, None), G._input_grad(g, w, None), G._weight_grad(g, h, False)
    assert torch.equal(G._forward(h, wt, None), out) and torch.equal(G._input_grad(g, wt, None), gh)
    wide = torch.empty(edges, width + 8, device=DEV)
    wide[:, 4:4 + width] = g
    assert torch.equal(G._input_grad(wide[:, 4:4 + width], w, None), gh)
    assert torch.equal(G._weight_grad(wide[:, 4:4 + width], h, False), gw)
    for pad in (1, 6):
        room = torch.full((edges, width + pad), 7.0, device=DEV)
        G._forward(h, w, room[:, :width])
        assert torch.equal(room[:, :width], out) and bool((room[:, width:] == 7.0).all())
    assert torch.equal(G._weight_grad(g, h, True).t(), gw)


def test_odd_width_forward():
    h, w, _ = _inputs(200, 131)
    _close(G._forward(h, w, None), h, w.t())


def test_non_finite_and_huge_values_as_in_float32():
    """Infinities, NaNs and values above the largest bf16: the float32 products' infinities and NaNs,
    the same finite values elsewhere."""
    h, w, g = _inputs(300, 100)
    w[7, 1] = 0.0
    h[5, 1], h[5, 3], h[77, 9], h[90, 2] = float("inf"), 2.0, 3.3999e38, float("nan")
    h[77, :9] = h[77, 10:] = 0.0
    g[5, 3], g[6, 9], g[8, 50] = float("-inf"), -3.3999e38, float("nan")
    for got, a, b in ((G._forward(h, w, None), h, w.t()), (G._input_grad(g, w, None), g, w),
                      (G._weight_grad(g, _inputs(300, 100)[0], False), g.t(), _inputs(300, 100)[0])):
        expect = a @ b
        assert torch.equal(torch.isnan(got), torch.isnan(expect)) and torch.equal(torch.isinf(got), torch.isinf(expect))
        keep = torch.isfinite(expect)
        assert torch.allclose(got[keep], expect[keep], rtol=1e-4, atol=1e-4)
    assert torch.isfinite(G._forward(h, w, None)[77]).any()


def test_rule_takes_the_three_forms_and_leaves_the_rest(monkeypatch):
    for name in ("FORWARD_ROWS", "FORWARD_RESULTS", "INPUT_GRAD_ROWS", "WEIGHT_GRAD_ROWS", "WEIGHT_GRAD_NARROW_ROWS"):
        monkeypatch.setattr(G, name, 256)
    h, w, g = _inputs(300, 144)
    for a, b in ((h, w.t()), (h, w.t().contiguous()), (g, w), (g, w.t().contiguous().t()), (g.t(), h), (h.t(), g)):
        got = G.product(a, b)
        assert got is not None and torch.equal(got, L._product(a, b))
        _close(got, a, b)
    odd = torch.empty(300 * 144 + 1, device=DEV)[1:].reshape(300, 144).copy_(g)     # not 16-byte aligned
    shared = [t[:, :132] for t in (g.reshape(-1)[:300 * 132].reshape(300, 132), g)]   # rows that share lines, and not
    assert G.product(shared[0], w[:132]) is None and G.product(shared[1], w[:132]) is not None
    room = torch.empty(300, 160, device=DEV)
    assert G.product(h, w.t(), room[:, :144]) is not None and G.product(h, w.t(), room[:, 8:152]) is None
    assert G.product(h, w[:136].t()) is None
    refused = [(odd, w), (h[:, :32], w[:, :32].t()), (h[:100], w.t()), (h, w[:64].t()), (h[::2], w.t()),
               (g[:, :131], w[:131]), (h.expand(300, 64)[:1].expand(300, 64), w.t()), (h.double(), w.double().t())]
    for a, b in refused:
        assert G.product(a, b) is None
    for a, b in refused[:-1]:
        assert torch.allclose(L._product(a, b), (a.double() @ b.double()).float(), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("rows,width,forward,weight", [
    (11718, 512, False, True), (11719, 512, True, True), (2048, 2928, False, True), (2048, 2944, True, True),
    (2047, 2944, False, False), (27000, 128, False, True), (4095, 636, False, False), (4095, 640, False, True),
    (4096, 128, False, True), (46000, 132, False, True)])
def test_lines_of_the_rule(rows, width, forward, weight):
    h, w, g = _inputs(rows, width)
    for a, b, taken in ((h, w.t(), forward), (g.t(), h, weight), (h.t(), g, weight), (g, w, False)):
        got = G.product(a, b)
        assert (got is not None) is taken
        _close(L._product(a, b), a, b)
