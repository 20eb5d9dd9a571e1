"""The 64-lane march at steps from far below to above a voxel, where the
sequence of steps crosses binades, ties or starts below the step, against the
one-lane oracle, bit for bit."""
import numpy as np
import pytest
import torch

from oracle import march as omarch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("step,res,cap", [
    (2.0 / 4096, 16, 0),              # 256 steps a voxel: skips past the 64 lanes
    (2.0 / 4096, 16, 100),
    (0.3, 32, 0),                     # steps above a voxel: every skip is one step
    (2.0 ** -8 + 2.0 ** -23, 32, 64), # ties at t in [2, 4): an addition moves by two amounts in turn
    (0.0067, 128, 65),
])
@pytest.mark.parametrize("n", [1, 67])
def test_march_steps_and_sequences_bitexact(dev, step, res, cap, n):
    from angelo_amd import functions as fn
    g = torch.Generator().manual_seed(res + n)
    o = torch.randn(n, 3, generator=g)
    o[::3] *= 0.3                                            # inside the box: t from 0
    o[1::3] = 3.1 * torch.nn.functional.normalize(o[1::3], dim=-1)   # binades at 2 and 4
    d = torch.nn.functional.normalize(0.4 * torch.randn(n, 3, generator=g) - o, dim=-1)
    d[::7, 0] = 0.0                                          # an axis without a crossing
    rays = torch.cat([o, d], -1).contiguous()
    grid = (torch.rand(res, res, res, generator=g) < 0.1).to(torch.uint8)
    grid[:, : res // 2] = 0                                  # a long empty half
    grid[:, -(res // 8):] = 1                                # runs of more than 64 samples
    aabb = [-1.0, -1.0, -1.0, 1.0, 1.0, 1.0]
    tn, tf = fn.ray_aabb(rays.to(dev), aabb)
    ridx, t0, t1, packed = fn.ray_marching(rays.to(dev), tn, tf, aabb, grid.to(dev), step, None, cap)
    on, of = omarch.ray_aabb(rays.numpy(), aabb)
    oi, o0, o1, oc = omarch.ray_marching(rays.numpy(), on, of, aabb, grid.numpy(), step, cap, None)
    assert np.array_equal(packed[:, 1].cpu().numpy(), oc)
    assert np.array_equal(ridx.cpu().numpy(), oi)
    assert np.array_equal(t0.cpu().numpy(), o0)
    assert np.array_equal(t1.cpu().numpy(), o1)
