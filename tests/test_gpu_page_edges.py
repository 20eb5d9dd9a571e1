"""The stand-alone grid's table gradient at the edges of a page (12288 pairs,
1536 points of eight pairs) against float64 sums of the pairs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1535, 1536, 1537, 3072, 3073])
def test_table_gradient_at_a_pages_edge(dev, n):
    from angelo_amd import descs
    from oracle import hashgrid as ohg
    from test_gpu_table_grad import _backward, _case, _pairs
    L, log2T, base, scale = 2, 14, 16, 2.0
    grid = descs.grid_desc(L, 2, log2T, base, scale)
    lt = ohg.level_table(L, base, scale, log2T, 2)
    x, dy = _case(L, log2T, base, scale, n, False, 11)
    got = _backward(x, dy, grid, L, dev).cpu().numpy().astype(np.float64)
    rows, v = _pairs(x, dy, lt, L)
    want = np.zeros((int(grid.n_entries), 2))
    mass = np.zeros_like(want)
    np.add.at(want, rows, v.astype(np.float64))
    np.add.at(mass, rows, np.abs(v).astype(np.float64))
    # one rounding of the sum, and each value's to 2^-35 of its row's largest
    assert (np.abs(got - want) <= 2.0 ** -24 * np.abs(want) + 2.0 ** -35 * mass + 1e-45).all()
