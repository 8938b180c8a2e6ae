"""Counting sort of the radius graph's atoms by bin, against the elementwise wrap and a stable sort:
coordinates on and beside bin edges and cell faces, bins given by the caller, sizes around a block."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("given", [False, True], ids=["fractional", "bins"])
@pytest.mark.parametrize("atoms,bins", [(1, (1, 1, 1)), (255, (3, 2, 5)), (257, (1, 7, 1)), (4099, (6, 6, 6))])
def test_bins(gpu, atoms, bins, given):
    from ictc_o3 import _lib
    generator = torch.Generator().manual_seed(atoms)
    frac = torch.rand(atoms, 3, generator=generator, dtype=torch.float64) * 6 - 3
    edges = torch.tensor([0.0, 1.0, -1.0, -1e-18, 1.0 - 2.0 ** -53, 1 / 3, 0.5, 2.0])
    frac[::3] = edges[torch.randint(0, 8, (len(frac[::3]), 3), generator=generator)].double()
    frac = frac.to(gpu)
    count = torch.tensor(bins, dtype=torch.float64, device=gpu)
    images = torch.floor(frac)
    wrapped = frac - images
    abin = torch.minimum(torch.floor(wrapped * count).clamp(min=0), count - 1).to(torch.int32)
    index = (abin[:, 0].long() * bins[1] + abin[:, 1]) * bins[2] + abin[:, 2]

    grid = _lib.CellGrid()
    grid.cutoff_sq = 1.0
    for a in range(3):
        grid.bins[a], grid.reach[a], grid.periodic[a] = bins[a], 1, 0 if given else 1
    nbins = bins[0] * bins[1] * bins[2]
    out_images = torch.empty(atoms, 3, dtype=torch.int64, device=gpu)
    out_wrapped = torch.empty_like(frac)
    out_bins = abin.clone() if given else torch.empty_like(abin)
    start = torch.zeros(nbins + 1, dtype=torch.int64, device=gpu)
    places = torch.empty(atoms, dtype=torch.int32, device=gpu)
    out = torch.full((atoms,), -1, dtype=torch.int64, device=gpu)
    lib, stream = _lib.lib(), _lib.stream_of(gpu)
    _lib.check(lib.ictc_hip_radius_graph_bins(ctypes.byref(grid), None if given else frac.data_ptr(), atoms,
                                              out_images.data_ptr(), out_wrapped.data_ptr(), out_bins.data_ptr(),
                                              start.data_ptr(), places.data_ptr(), stream), "bins")
    start = torch.cumsum(start, 0)
    _lib.check(lib.ictc_hip_radius_graph_bin_atoms(ctypes.byref(grid), out_bins.data_ptr(), places.data_ptr(),
                                                   start.data_ptr(), atoms, out.data_ptr(), stream), "bin_atoms")
    if not given:
        assert torch.equal(out_images, images.long()) and torch.equal(out_wrapped, wrapped)
        assert torch.equal(out_bins, abin)
    assert torch.equal(start[1:], torch.bincount(index, minlength=nbins).cumsum(0)) and int(start[0]) == 0
    # each bin's atoms, in any order within the bin
    assert torch.equal(index[out], index.sort().values)
    assert torch.equal(out.sort().values, torch.arange(atoms, device=gpu))
