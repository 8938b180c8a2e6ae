"""The contraction's weight gradients summed in one pass over the species-ordered nodes: equal to the
per-node features summed in float64, for empty and single-node species, ranges that split a species, partial
channel chunks and plans at both sides of the column limit; bit-identical from run to run.

Tolerance: a species' sum over n nodes is three nested fp32 sums (a range's nodes, then the ranges), within
n * 2^-24 of the sum of the features' magnitudes at worst; the features themselves are compared as the
kernel's own float32 values."""
import pytest
import torch

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from ictc_o3 import _lib  # noqa: E402
from ictc_o3.backends.hip import symmetric_contraction as S  # noqa: E402

DEV = torch.device("cuda", 0)


def _features(plan, x, species, go, t):
    phi = torch.empty(x.shape[0], plan.ktot, plan.channels, device=DEV)
    lib, p = _lib.lib(), _lib.ptr
    args = (plan.lmax, plan.target_lmax, plan.correlation, plan.channels, p(x), p(species), plan.num_elements, p(go))
    if t is None:
        st = lib.ictc_hip_sc_weight_features(*args, p(phi), x.shape[0], _lib.stream_of(DEV))
    else:
        st = lib.ictc_hip_sc_weight_features_jvp(*args, p(t), p(phi), x.shape[0], _lib.stream_of(DEV))
    assert st == 0
    return phi.double()


@pytest.mark.parametrize("plan_args,channels,elements,nodes", [
    ((3, 1, 3), 128, 10, 1543), ((3, 0, 3), 64, 3, 257), ((2, 2, 3), 24, 89, 300), ((1, 1, 2), 130, 1, 5000),
    ((1, 1, 3), 64, 4, 301), ((2, 0, 3), 32, 9, 1200), ((2, 0, 3), 32, 9, 1201),    # the shortest ranges' lines
    ((0, 0, 1), 1, 2, 1), ((3, 3, 2), 96, 5, 33), ((3, 1, 3), 64, 7, 40000)])
@pytest.mark.parametrize("tangent", [False, True])
def test_weight_gradient_matches_summed_features(plan_args, channels, elements, nodes, tangent):
    plan = S.ContractionPlan(*plan_args, channels, elements)
    gen = torch.Generator().manual_seed(nodes)
    x, t = (torch.randn(nodes, plan.in_width, generator=gen).to(DEV) for _ in range(2))
    go = torch.randn(nodes, plan.out_width, generator=gen).to(DEV)
    species = torch.randint(0, elements, (nodes,), generator=gen)
    if elements > 4:
        species[species == 2] = 3                       # a species without nodes
        species[species == 4] = 0
        species[nodes // 2] = 4                         # one with a single node
    species = species.to(DEV)
    t = t if tangent else None
    got = S._weight_grad_fused(plan, x, species, go, t)
    assert got is not None
    assert torch.equal(got, S._weight_grad_fused(plan, x, species, go, t))
    phi = _features(plan, x, species, go, t)
    want, size = (torch.zeros(elements, plan.ktot, channels, dtype=torch.float64, device=DEV).index_add_(0, species, v)
                  for v in (phi, phi.abs()))
    per_species = torch.bincount(species, minlength=elements).double()[:, None, None]
    assert bool(((got.double() - want).abs() <= (per_species + 1) * 2.0 ** -24 * size).all())
    full = S._weight_grad(plan, x, species, go) if t is None else S._weight_grad_jvp(plan, x, species, go, t)
    assert torch.equal(full, got)


def test_no_nodes_and_wider_plans():
    plan = S.ContractionPlan(3, 1, 3, 32, 4)
    empty = torch.empty(0, dtype=torch.int64, device=DEV)
    got = S._weight_grad_fused(plan, torch.empty(0, plan.in_width, device=DEV), empty,
                               torch.empty(0, plan.out_width, device=DEV))
    assert got.shape == (4, plan.ktot, 32) and not got.any()
    wide = S.ContractionPlan(3, 2, 3, 32, 4)            # 159 columns: features and a product
    x = torch.randn(50, wide.in_width, device=DEV)
    go = torch.randn(50, wide.out_width, device=DEV)
    species = torch.arange(50, device=DEV) % 4
    assert S._weight_grad_fused(wide, x, species, go) is None
    phi = _features(wide, x, species, go, None)
    want = torch.zeros(4, wide.ktot, 32, dtype=torch.float64, device=DEV).index_add_(0, species, phi)
    assert torch.allclose(S._weight_grad(wide, x, species, go).double(), want, rtol=1e-4, atol=1e-3)
