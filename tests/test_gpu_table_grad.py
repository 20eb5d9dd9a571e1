"""The table-gradient reduction against float64 sums of the very pairs it is
given (am_hashgrid_bwd: eight (row, w * g) pairs per level and point, the rows
and fp32 weights from the oracle)."""
import numpy as np
import pytest
import torch

from oracle import hashgrid as ohg

pytestmark = pytest.mark.gpu


def _case(L, log2T, base, scale, n, cluster, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.rand(n, 3, generator=g)
    if cluster:   # many points in one cell: rows with many pairs, sliced buckets
        x = 0.37 + 0.02 * x
    dy = torch.randn(n, 2 * L, generator=g) * torch.pow(10.0, -4 * torch.rand(n, 1, generator=g))
    return x, dy


def _pairs(x, dy, lt, active):
    """Level-offset rows and fp32 pair values [n * active * 8 (, 2)]."""
    _, _, idx, w = ohg.corners(x.numpy(), lt)
    rows = idx[:, :active].astype(np.int64) + lt.offset[None, :active, None].astype(np.int64)
    g = dy.numpy().reshape(x.shape[0], lt.n_levels, 1, 2)[:, :active]
    v = (w[:, :active, :, None] * g).astype(np.float32)   # one fp32 product each
    return rows.reshape(-1), v.reshape(-1, 2)


def _backward(x, dy, grid, active, dev):
    from angelo_amd.functions import hashgrid_encode
    t = torch.zeros(int(grid.n_entries), 2, device=dev, requires_grad=True)
    out = hashgrid_encode(x.to(dev), t, grid, active)
    return torch.autograd.grad(out, t, dy.to(dev))[0]


@pytest.mark.parametrize("L,log2T,base,scale,active,n,cluster", [
    (1, 10, 4, 2.0, 1, 1, False),            # eight pairs
    (2, 13, 16, 2.0, 2, 768, False),         # a page's 6144 pairs a level, one full bucket
    (3, 14, 16, 2.0, 2, 769, False),         # one pair set more; a level without pairs
    (4, 19, 32, 1.5, 4, 30011, False),       # ragged pages, buckets cut by a level's end
    (2, 21, 128, 4.0, 2, 20000, False),      # the most buckets of a level
    (2, 15, 16, 2.0, 2, 60000, True),        # sliced buckets, long runs of one row
    (1, 22, 300, 2.0, 1, 20000, False),      # a level past 2^21 rows: the sorted form
])
def test_table_gradient_is_the_exact_sum_of_its_pairs(dev, L, log2T, base, scale, active, n,
                                                      cluster):
    from angelo_amd import descs
    grid = descs.grid_desc(L, 2, log2T, base, scale)
    lt = ohg.level_table(L, base, scale, log2T, 2)
    x, dy = _case(L, log2T, base, scale, n, cluster, 3)
    got = _backward(x, dy, grid, active, dev)
    assert torch.equal(got, _backward(x, dy, grid, active, dev))   # the same bits again
    rows, v = _pairs(x, dy, lt, active)
    want = np.zeros((int(grid.n_entries), 2))
    mass = np.zeros_like(want)
    np.add.at(want, rows, v.astype(np.float64))
    np.add.at(mass, rows, np.abs(v).astype(np.float64))
    err = np.abs(got.cpu().numpy().astype(np.float64) - want)
    if log2T <= 21:
        # one rounding of the sum, and each value's to 2^-35 of its row's largest
        assert (err <= 2.0 ** -24 * np.abs(want) + 2.0 ** -35 * mass + 1e-45).all()
    else:   # float sums: 2^-24 of the partial sums an addition
        assert (err <= 1e-5 * mass).all()


def test_table_gradient_keeps_infinities_and_nan_in_their_rows(dev):
    """A row with a non-finite pair gets the class of its sum per feature, and
    every other row its ordinary sum."""
    from angelo_amd import descs
    L, log2T, base, scale, n = 2, 14, 16, 2.0, 5000
    grid = descs.grid_desc(L, 2, log2T, base, scale)
    lt = ohg.level_table(L, base, scale, log2T, 2)
    x, dy = _case(L, log2T, base, scale, n, False, 5)
    dy[7, 0], dy[11, 1], dy[12, 3], dy[40, 2] = float("inf"), float("-inf"), float("nan"), 3e38
    got = _backward(x, dy, grid, L, dev).cpu().numpy()
    rows, v = _pairs(x, dy, lt, L)
    want = np.zeros((int(grid.n_entries), 2))
    np.add.at(want, rows, v.astype(np.float64))
    with np.errstate(over="ignore"):
        want32 = want.astype(np.float32)
    bad = ~np.isfinite(want32)
    assert bad.any()
    assert np.array_equal(np.isnan(got), np.isnan(want32))
    assert np.array_equal(got[bad & ~np.isnan(want32)], want32[bad & ~np.isnan(want32)])
    np.testing.assert_allclose(got[~bad], want32[~bad], rtol=1e-6, atol=1e-30)
