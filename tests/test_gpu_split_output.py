"""MLP gradients of the difference form, whose offset evaluations take the SDF
row alone through the output layer, against the same differences built from
single evaluations."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 17, 1000])
@pytest.mark.parametrize("kw", [dict(L=8, log2T=15, base=16, scale=1.5, feature_dim=4),
                                dict(L=16, log2T=16, base=32, scale=1.3195079107728942),
                                dict(L=8, log2T=15, base=16, scale=1.5, geo_hidden=2)])
def test_offset_gradients_equal_single_evaluations(dev, kw, n):
    from test_gpu_pipeline import _field_model
    model = _field_model(dev, **kw)
    geo = model.geometry
    geo._finite_difference_eps = eps = 0.1
    g = torch.Generator().manual_seed(n)
    pts = ((torch.rand(n, 3, generator=g) * 2 - 1) * 0.8).to(dev)
    c = torch.randn(n, 3, generator=g).to(dev)
    params = list(geo.network.parameters())
    sdf, grad = geo.fused(pts, with_grad=True)[:2]
    got = torch.autograd.grad((grad * c).sum() + sdf.sum(), params)
    loss = geo.fused(pts, with_grad=False)[0].sum()
    for d in range(3):
        step = torch.zeros(3, device=dev)
        step[d] = eps
        hi, lo = (geo.fused(p, with_grad=False)[0] for p in (pts + step, pts - step))
        loss = loss + ((hi - lo) * (0.5 / eps) * c[:, d]).sum()
    want = torch.autograd.grad(loss, params)
    for a, b in zip(got, want):   # fp32 sums of 13 n terms in another order
        torch.testing.assert_close(a, b, rtol=1e-4, atol=2e-5 * float(b.abs().max()) + 1e-7)
