"""Table gradients of grid descriptors whose levels do not follow one another
from row 0: another order, gaps, rows that two levels share.  Every row of the
gradient is written, rows without a level with zeros."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

L, LOG2T, BASE, SCALE = 3, 13, 12, 1.7


def _grid(layout):
    """The descriptor and, for each of its rows' levels, the first row."""
    from angelo_amd import descs
    grid = descs.grid_desc(L, 2, LOG2T, BASE, SCALE)
    size = [int(s) for s in grid.size[:L]]
    if layout == "reversed":
        first, rows = [size[1] + size[2], size[2], 0], sum(size)
    elif layout == "gaps":
        first, rows = [8, 8 + size[0] + 1000, 8 + size[0] + 1000 + size[1]], sum(size) + 1108
    elif layout == "shared":
        first, rows = [0, 0, size[1]], size[1] + size[2]
    else:
        first, rows = [0, size[0], size[0] + size[1]], sum(size) + 16   # rows after the last level
    for l in range(L):
        grid.offset[l] = first[l]
    grid.n_entries = rows
    return grid, first


@pytest.mark.parametrize("layout", ["reversed", "gaps", "shared", "tail"])
def test_hash_grid_gradient_of_other_layouts(dev, layout):
    from angelo_amd.functions import hashgrid_encode
    from oracle import hashgrid as ohg
    grid, first = _grid(layout)
    lt = ohg.level_table(L, BASE, SCALE, LOG2T, 2)
    g = torch.Generator().manual_seed(21)
    n = 2000
    x, dy = torch.rand(n, 3, generator=g), torch.randn(n, 2 * L, generator=g)
    t = torch.zeros(int(grid.n_entries), 2, device=dev, requires_grad=True)
    torch.full((2 * t.numel(),), float("nan"), device=dev)   # what the next block may hold
    got = torch.autograd.grad(hashgrid_encode(x.to(dev), t, grid, L), t, dy.to(dev))[0]
    _, _, idx, w = ohg.corners(x.numpy(), lt)
    rows = idx.astype(np.int64) + np.array(first)[None, :, None]
    v = (w[..., None] * dy.numpy().reshape(n, L, 1, 2)).astype(np.float32)
    want, mass = np.zeros((t.shape[0], 2)), np.zeros((t.shape[0], 2))
    np.add.at(want, rows.reshape(-1), v.reshape(-1, 2).astype(np.float64))
    np.add.at(mass, rows.reshape(-1), np.abs(v.reshape(-1, 2)).astype(np.float64))
    err = np.abs(got.cpu().numpy().astype(np.float64) - want)
    assert (err <= 1e-5 * mass).all()   # fp32 sums; rows without a pair are zero


@pytest.mark.parametrize("layout", ["reversed", "gaps", "shared", "tail"])
def test_field_gradient_of_other_layouts(dev, layout):
    """The field's backward against its atomic form, which adds each pair into
    its row."""
    from angelo_amd import _native as nat
    from test_gpu_pipeline import _field_model
    geo = _field_model(dev, L=L, log2T=LOG2T, base=BASE, scale=SCALE).geometry
    grid, _ = _grid(layout)
    module = geo.grid_module
    module.grid = grid
    g = torch.Generator().manual_seed(22)
    module.params = torch.nn.Parameter(
        ((torch.rand(int(grid.n_entries) * 2, generator=g) - 0.5) * 0.1).to(dev))
    n = 1500
    pts = ((torch.rand(n, 3, generator=g) * 2 - 1) * 0.9).to(dev)
    randn = torch.randn(n, 3, generator=g).to(dev)
    got = {}
    for atomic in (0, 1):
        nat.set_flag("table_atomic", atomic)
        try:
            geo.zero_grad()
            sdf, grad, normal, feature, lap = geo.fused(pts, True, True, randn)
            (sdf.sum() + grad.square().sum() + lap.sum() + feature.sum()).backward()
            got[atomic] = module.params.grad.clone()
        finally:
            nat.set_flag("table_atomic", 0)
    nat.sdf_bwd_check()
    top = float(got[1].abs().max())
    assert top > 0
    # fp32 sums of up to a few hundred terms per row in another order
    torch.testing.assert_close(got[0], got[1], rtol=1e-4, atol=1e-6 * top)
