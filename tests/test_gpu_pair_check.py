"""The field backward's check that its emission puts as many table-gradient
pairs as its count pass found.  One count is moved from the host; every kernel
runs to its end inside its arrays."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _gradient(geo, pts, randn):
    geo.zero_grad()
    sdf, grad, normal, feature, lap = geo.fused(pts, True, True, randn)
    (sdf.sum() + grad.square().sum() + lap.sum() + feature.sum()).backward()
    return geo.grid_module.params.grad.clone()


@pytest.mark.parametrize("sync_free", [False, True])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("shift", [4, 60, -4])
def test_emission_reports_a_count_that_does_not_fit(dev, shift, mixed, sync_free):
    from angelo_amd import _native as nat, functions as fn
    from test_gpu_pipeline import _field_model
    geo = _field_model(dev, L=8, log2T=15, base=16, scale=1.5).geometry
    if mixed:
        geo.set_precision("mixed")
    g = torch.Generator().manual_seed(9)
    n = 150   # a page a level
    pts = ((torch.rand(n, 3, generator=g) * 2 - 1) * 0.9).to(dev)
    randn = torch.randn(n, 3, generator=g).to(dev)
    fn.set_sdf_backward(sync_free=sync_free)
    try:
        want = _gradient(geo, pts, randn)
        nat.sdf_bwd_check()
        nat.set_flag("sdf_bwd_count_shift", shift)
        try:
            got = _gradient(geo, pts, randn)
            with pytest.raises(RuntimeError, match="mismatch"):
                nat.sdf_bwd_check()
        finally:
            nat.set_flag("sdf_bwd_count_shift", 0)
        assert bool(torch.isfinite(got).all())
        if shift > 0:   # fewer pairs put than counted: all of them, and nothing else
            assert torch.equal(got, want)
        assert torch.equal(_gradient(geo, pts, randn), want)
        nat.sdf_bwd_check()
    finally:
        fn.set_sdf_backward(sync_free=False)


@pytest.mark.parametrize("cut", [1, 5, 1 << 20])
def test_emission_stays_inside_short_arrays(dev, cut):
    """Arrays of fewer pages than the emission needs: reported, and the pages
    that are there are all that the reduction reads."""
    from angelo_amd import _native as nat
    from test_gpu_pipeline import _field_model
    geo = _field_model(dev, L=8, log2T=15, base=16, scale=1.5).geometry
    g = torch.Generator().manual_seed(10)
    n = 2100   # three units a level, several pages each
    pts = ((torch.rand(n, 3, generator=g) * 2 - 1) * 0.9).to(dev)
    randn = torch.randn(n, 3, generator=g).to(dev)
    want = _gradient(geo, pts, randn)
    nat.sdf_bwd_check()
    nat.set_flag("sdf_bwd_page_cut", cut)
    try:
        got = _gradient(geo, pts, randn)
        with pytest.raises(RuntimeError, match="mismatch"):
            nat.sdf_bwd_check()
    finally:
        nat.set_flag("sdf_bwd_page_cut", 0)
    coarse = int(geo.grid_module.grid.offset[1]) * 2
    if cut == 1:   # the last unit's pages are missing: the coarsest level keeps its bits
        assert torch.equal(got.view(-1)[:coarse], want.view(-1)[:coarse])
    if cut == 1 << 20:
        assert not bool(got.any())
    assert bool(torch.isfinite(got).all())
    assert torch.equal(_gradient(geo, pts, randn), want)
    nat.sdf_bwd_check()
