"""The reduction's work units: buckets cut by their own load where points
crowd, buckets without pairs, few pages (counted by the plan itself) and many,
against float64 sums of the pairs."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,log2T,base,scale,active,n,width", [
    (2, 21, 128, 4.0, 2, 500, 0.004),      # a page a level; 500 buckets without pairs
    (2, 21, 128, 4.0, 2, 9300, 0.004),     # a bucket just past a unit and a half (73,728 pairs)
    (2, 21, 128, 4.0, 2, 25000, 0.004),    # a few slices
    (2, 21, 128, 4.0, 2, 60000, 0.004),    # many slices, merged by four waves
    (1, 6, 4, 2.0, 1, 70001, 1.0),         # one bucket of 64 rows
    (5, 17, 16, 2.0, 4, 30011, 0.1),       # a last bucket cut by its level's end, an empty level
])
def test_buckets_are_cut_by_their_own_load(dev, L, log2T, base, scale, active, n, width):
    from angelo_amd import descs
    from oracle import hashgrid as ohg
    from test_gpu_table_grad import _backward, _pairs
    grid = descs.grid_desc(L, 2, log2T, base, scale)
    lt = ohg.level_table(L, base, scale, log2T, 2)
    g = torch.Generator().manual_seed(n)
    x = 0.3 * (1 - width) + width * torch.rand(n, 3, generator=g)
    dy = torch.randn(n, 2 * L, generator=g) * torch.pow(10.0, -4 * torch.rand(n, 1, generator=g))
    got = _backward(x, dy, grid, active, dev)
    assert torch.equal(got, _backward(x, dy, grid, active, dev))   # the same bits again
    rows, v = _pairs(x, dy, lt, active)
    want = np.zeros((int(grid.n_entries), 2))
    mass = np.zeros_like(want)
    np.add.at(want, rows, v.astype(np.float64))
    np.add.at(mass, rows, np.abs(v).astype(np.float64))
    err = np.abs(got.cpu().numpy().astype(np.float64) - want)
    # one rounding of the sum, and each value's to 2^-42 of its row's largest
    # (at most 2^19 pairs a unit), 2^-35 of the values' mean at their spread
    assert (err <= 2.0 ** -24 * np.abs(want) + 2.0 ** -35 * mass + 1e-45).all()
