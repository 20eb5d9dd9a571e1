"""The paged emission of the field's table-gradient pairs against the atomic
form, which shares no emitting code with it: each evaluation is classified and
merged by the general rule, in any position, and added into its row at once."""
import pytest
import torch

pytestmark = pytest.mark.gpu

NGP = dict(L=16, log2T=19, base=32, scale=1.3195079107728942)


def _table_gradient(model, pts, randn, grad, laplace, atomic, normalised=True):
    from angelo_amd import _native as nat
    geo = model.geometry
    nat.set_flag("table_atomic", atomic)
    try:
        model.zero_grad()
        out = list(geo.fused(pts, grad, laplace, randn))
        if not normalised:
            out[2] = out[4] = None   # laplace divides by the gradient's length
        loss = sum((o * torch.linspace(0.5, 1.5, o.numel(), device=o.device).view_as(o)).sum()
                   for o in out if o is not None)
        loss.backward()
        torch.cuda.synchronize()
    finally:
        nat.set_flag("table_atomic", 0)
    nat.sdf_bwd_check()
    return model.geometry.grid_module.params.grad.clone()


@pytest.mark.parametrize("kw,n,eps,reach,grad,laplace,start,mixed", [
    (NGP, 1, None, 0.9, True, True, None, False),        # one sample
    (NGP, 1023, None, 0.9, True, True, None, False),     # a unit's edges
    (NGP, 1025, None, 0.9, True, True, None, False),
    (NGP, 3000, 0.07, 0.9, True, True, None, False),     # offsets past the next cell: 8 corners each
    (NGP, 3000, 0.02, 0.9, True, True, None, False),     # both ways, by level
    (NGP, 3000, None, 1.3, True, True, None, False),     # points outside the box
    (NGP, 20000, None, 0.02, True, True, None, False),   # all in few cells: long merges
    (NGP, 3000, None, 0.9, True, True, 3, False),        # few active levels
    (NGP, 3000, None, 0.9, True, False, None, False),
    (NGP, 3000, None, 0.9, False, False, None, False),   # the base evaluation alone
    (dict(NGP, grad_type="analytic"), 3000, None, 0.9, True, True, None, False),
    (NGP, 3000, None, 0.9, True, True, None, True),      # fp16 pairs
    (dict(L=5, log2T=21, base=64, scale=2.0), 3000, None, 0.9, True, True, None, False),
])
def test_paged_table_gradient_matches_the_atomic_form(dev, kw, n, eps, reach, grad, laplace, start,
                                                      mixed):
    from test_gpu_pipeline import _field_model
    model = _field_model(dev, **kw)
    if mixed:
        model.geometry.set_precision("mixed")
    if eps is not None:
        model.geometry._finite_difference_eps = eps
    if start is not None:
        model.geometry.grid_module.active_levels = start
    g = torch.Generator().manual_seed(n)
    pts = ((torch.rand(n, 3, generator=g) * 2 - 1) * reach).to(dev)
    randn = torch.randn(n, 3, generator=g).to(dev)
    # outside the box clamped offsets give zero gradients, and what divides by
    # their length has gradients (1e14 and cancelling) that leave float sums in
    # any order no digits: two runs of the atomic form differ by their own size
    normalised = reach < 1.0
    got = _table_gradient(model, pts, randn, grad, laplace, 0, normalised)
    assert torch.equal(got, _table_gradient(model, pts, randn, grad, laplace, 0, normalised))
    want = _table_gradient(model, pts, randn, grad, laplace, 1, normalised)
    assert bool(torch.isfinite(want).all()) and float(want.abs().max()) > 0
    top = float(want.abs().max())
    if mixed:   # each pair rounded to 11 bits; a row's sum of magnitudes within 8 of the largest sum
        torch.testing.assert_close(got, want, rtol=2.0 ** -10, atol=8 * 2.0 ** -11 * top)
    else:       # fp32 sums of up to a few hundred terms per row in another order
        torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-6 * top)
