"""The spatial order's counting passes at the edges of tiles and blocks."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bits", [(1, 5), (63, 1), (1024, 3), (1025, 5), (262145, 5),
                                    (262144, 6), (524289, 10)])
@pytest.mark.parametrize("spread", [True, False])
def test_order_is_the_stable_sort_of_the_keys(dev, n, bits, spread):
    from angelo_amd import functions
    g = torch.Generator().manual_seed(n)
    pts = torch.rand(n, 3, generator=g) * 2.4 - 1.2
    if not spread:   # few cells: digits with most of a tile
        pts = torch.round(pts * 1.5) * 0.4
    if n > 100:
        pts[7, 1] = float("nan")
    perm, inv = functions.spatial_order(pts.to(dev), 1.0, bits)
    cells = 1 << bits
    u = ((pts + 1.0) * 0.5).nan_to_num(0.0).clamp(0, 1)
    q = (u * cells).floor().clamp(max=cells - 1).long().numpy()
    key = np.zeros(n, np.int64)
    for b in range(bits):
        for d in range(3):
            key |= ((q[:, d] >> b) & 1) << (3 * b + (2 - d))
    ref = np.argsort(key, kind="stable")
    assert np.array_equal(perm.cpu().numpy(), ref)
    assert np.array_equal(inv.cpu().numpy()[ref], np.arange(n))
