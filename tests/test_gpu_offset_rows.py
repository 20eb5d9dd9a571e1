"""Offset evaluations from the centre's rows against single evaluations of the
offset points, which gather all their rows: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

NGP = dict(L=16, log2T=19, base=32, scale=1.3195079107728942)


@pytest.mark.parametrize("kw,n,eps,reach,active,precision", [
    (NGP, 1, None, 0.9, None, "fp32"),
    (NGP, 3001, None, 0.9, None, "fp32"),
    (NGP, 3001, 0.02, 0.9, None, "fp32"),    # eps above the fine levels' cells
    (NGP, 3001, 0.2, 0.9, None, "fp32"),     # above nearly all
    (NGP, 3001, 1e-5, 0.9, None, "fp32"),    # mostly the centre's cell
    (NGP, 3001, None, 1.02, None, "fp32"),   # samples at and beyond the box's faces
    (NGP, 3001, None, 0.9, 5, "fp32"),
    (NGP, 3001, 0.02, 1.02, None, "mixed"),
    (dict(L=8, log2T=15, base=16, scale=1.5), 3001, None, 1.02, None, "fp32"),
    (dict(L=6, log2T=21, base=64, scale=2.0, geo_hidden=2), 3001, None, 0.9, None, "fp32"),
])
def test_differences_equal_single_evaluations(dev, kw, n, eps, reach, active, precision):
    from test_gpu_pipeline import _field_model
    model = _field_model(dev, **kw)
    geo = model.geometry
    geo.set_precision(precision)
    if eps is not None:
        geo._finite_difference_eps = eps
    if active is not None:
        geo.grid_module.active_levels = active
    g = torch.Generator().manual_seed(n)
    pts = (torch.rand(n, 3, generator=g) * 2 - 1) * reach
    pts[: n // 4] = (pts[: n // 4] * 40).round() / 40        # on cell faces of dense levels
    pts = pts.to(dev)
    e = torch.tensor(float(geo._sdf_desc(True, False).fd_eps), dtype=torch.float32)
    inv = torch.ones((), dtype=torch.float32) / e
    with torch.no_grad():
        sdf, grad = geo.fused(pts, with_grad=True)[:2]
        assert torch.equal(sdf, geo.fused(pts, with_grad=False)[0])
        for d in range(3):
            step = torch.zeros(3, device=dev)
            step[d] = float(e)
            r = geo.radius
            hi, lo = ((p.clamp(-r, r)) for p in (pts + step, pts - step))
            diff = geo.fused(hi, with_grad=False)[0] - geo.fused(lo, with_grad=False)[0]
            assert torch.equal(grad[:, d], (0.5 * diff) * float(inv)), d
