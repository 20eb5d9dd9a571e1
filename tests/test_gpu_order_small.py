"""The spatial order of small batches (one block, all passes in LDS) and at the
edge to the general passes; its keys and stability from numpy."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 1023, 1024, 1025, 4095, 4096, 4097])
@pytest.mark.parametrize("bits", [1, 3, 5, 6, 10])
@pytest.mark.parametrize("spread", [True, False])
def test_order_of_small_batches(dev, n, bits, spread):
    from angelo_amd import functions
    g = torch.Generator().manual_seed(n + bits)
    pts = torch.rand(n, 3, generator=g) * 2.4 - 1.2
    if not spread:   # few cells: digits with most of a tile
        pts = torch.round(pts * 1.5) * 0.4
    perm, inv = functions.spatial_order(pts.to(dev), 1.0, bits)
    cells = 1 << bits
    u = ((pts + 1.0) * 0.5).clamp(0, 1)
    q = (u * cells).floor().clamp(max=cells - 1).long().numpy()
    key = np.zeros(n, np.int64)
    for b in range(bits):
        for d in range(3):
            key |= ((q[:, d] >> b) & 1) << (3 * b + (2 - d))
    ref = np.argsort(key, kind="stable")
    assert np.array_equal(perm.cpu().numpy(), ref)
    assert np.array_equal(inv.cpu().numpy()[ref], np.arange(n))
