"""The SDF backward's worst-case workspace (host arithmetic, no device)."""
import pytest


@pytest.mark.parametrize("rows", [15, 19, 21])
def test_worst_case_workspace_follows_the_samples(rows):
    from angelo_amd import _native as nat, descs
    grid = descs.grid_desc(16, 2, rows, 32, 1.3195079107728942)
    m = descs.mlp_desc(35, 16, 1)
    s = nat.SdfDesc()
    s.radius, s.fd_eps, s.with_grad, s.with_laplace, s.active_levels = 1.0, 1e-3, 1, 1, 16

    def size(n):
        return nat.load().am_sdf_bwd_workspace_size(nat.sptr(grid), nat.sptr(m), nat.sptr(s), n)

    # at most 108 pairs a sample and level: a call of a few samples does not pay
    # for a whole unit of 1024
    assert 0 < size(1) < 8 << 20
    assert size(64) < 8 << 20
    sizes = [size(n) for n in (1, 15, 16, 64, 75, 76, 300, 1023, 1024, 1025, 4096, 20011)]
    assert sizes == sorted(sizes)
