"""Marching many rays of few steps, or of many steps a cell (four lanes to a
ray), against the same rays in smaller calls (a wave to a ray), bit for bit,
and against the oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("step,res,cap,n,part", [
    (0.3, 32, 0, 18500, 18000),        # every skip is one step; just above the rule's rays
    (0.1, 64, 0, 70001, 40000),
    (0.1, 64, 7, 70001, 40000),        # a cap that rays reach: staged
    (2.0 * 3 ** 0.5 / 79.9, 16, 0, 128003, 100000),   # just within 80 steps
    (2.0 / 16 / 8.1, 16, 0, 65537, 65536),            # just above 8 steps a cell
    (2.0 / 4 / 40, 4, 20, 65541, 65536),
])
def test_march_forms_agree(dev, step, res, cap, n, part):
    from angelo_amd import functions as fn
    from oracle import march as omarch
    g = torch.Generator().manual_seed(res)
    o = torch.randn(n, 3, generator=g)
    o[::3] *= 0.3                                            # inside the box: t from 0
    d = torch.nn.functional.normalize(0.4 * torch.randn(n, 3, generator=g) - o, dim=-1)
    d[::7, 0] = 0.0                                          # an axis without a crossing
    rays = torch.cat([o, d], -1).contiguous()
    grid = (torch.rand(res, res, res, generator=g) < 0.2).to(torch.uint8)
    grid[:, -1:] = 1
    aabb = [-1.0, -1.0, -1.0, 1.0, 1.0, 1.0]
    tn, tf = fn.ray_aabb(rays.to(dev), aabb)
    ridx, t0, t1, packed = fn.ray_marching(rays.to(dev), tn, tf, aabb, grid.to(dev), step, None, cap)
    parts = [fn.ray_marching(rays[q].contiguous().to(dev), tn[q].contiguous(), tf[q].contiguous(), aabb,
                             grid.to(dev), step, None, cap)
             for q in (slice(0, part), slice(part, n))]
    assert torch.equal(packed[:, 1], torch.cat([p[3][:, 1] for p in parts]))
    assert torch.equal(t0, torch.cat([p[1] for p in parts]))
    assert torch.equal(t1, torch.cat([p[2] for p in parts]))
    assert torch.equal(ridx, torch.cat([parts[0][0], parts[1][0] + part]))
    on, of = omarch.ray_aabb(rays.numpy(), aabb)
    oi, o0, o1, oc = omarch.ray_marching(rays.numpy(), on, of, aabb, grid.numpy(), step, cap, None)
    assert np.array_equal(packed[:, 1].cpu().numpy(), oc)
    assert np.array_equal(ridx.cpu().numpy(), oi)
    assert np.array_equal(t0.cpu().numpy(), o0)
    assert np.array_equal(t1.cpu().numpy(), o1)
