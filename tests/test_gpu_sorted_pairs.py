"""The field backward's sorted form (a level past 2^21 rows): counted and
worst-case pair arrays against each other, bit for bit, and against the atomic
form, which adds the same merged pairs into their rows without arrays."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _gradients(geo, pts, randn, grad, laplace, atomic=0, sync_free=False):
    from angelo_amd import _native as nat, functions as fn
    nat.set_flag("table_atomic", atomic)
    fn.set_sdf_backward(sync_free=sync_free)
    try:
        geo.zero_grad()
        out = geo.fused(pts, grad, laplace, randn)
        sum((o * torch.linspace(0.5, 1.5, o.numel(), device=o.device).view_as(o)).sum()
            for o in out if o is not None).backward()
        torch.cuda.synchronize()
    finally:
        nat.set_flag("table_atomic", 0)
        fn.set_sdf_backward(sync_free=False)
    nat.sdf_bwd_check()
    return [p.grad.clone() for p in geo.parameters()]


@pytest.mark.parametrize("kw,n,grad,laplace,mixed", [
    (dict(L=1, base=300), 1, True, True, False),                  # one sample
    (dict(L=1, base=300), 3001, True, True, False),               # a ragged tile of 16 and group of 64
    (dict(L=2, base=200, scale=1.5), 1039, True, True, True),     # fp16 pairs
    (dict(L=2, base=200, scale=1.5), 3001, True, False, False),
    (dict(L=2, base=16, scale=16.0), 2000, False, False, False),  # a coarse level beside it
    (dict(L=2, base=200, scale=1.5, grad_type="analytic"), 1039, True, True, False),
    (dict(L=9, base=200, scale=1.1), 515, True, True, False),     # four level slots a lane group
])
def test_sorted_table_gradient(dev, kw, n, grad, laplace, mixed):
    from test_gpu_pipeline import _field_model
    geo = _field_model(dev, log2T=22, **kw).geometry
    if mixed:
        geo.set_precision("mixed")
    g = torch.Generator().manual_seed(n)
    pts = ((torch.rand(n, 3, generator=g) * 2 - 1) * 0.9).to(dev)
    randn = torch.randn(n, 3, generator=g).to(dev)
    got = _gradients(geo, pts, randn, grad, laplace)
    for a, b in zip(got, _gradients(geo, pts, randn, grad, laplace, sync_free=True)):
        assert torch.equal(a, b)
    want = _gradients(geo, pts, randn, grad, laplace, atomic=1)
    names = [k for k, _ in geo.named_parameters()]
    for k, a, b in zip(names, got, want):
        assert bool(torch.isfinite(b).all()), k
        if b.numel() != geo.grid_module.params.numel():
            assert torch.equal(a, b), k   # no MLP gradient passes through the table's sums
            continue
        top = float(b.abs().max())
        assert top > 0
        if mixed:   # each pair rounded to 11 bits; a row's sum of magnitudes within 8 of the largest
            torch.testing.assert_close(a, b, rtol=2.0 ** -10, atol=8 * 2.0 ** -11 * top)
        else:       # fp32 sums of up to a few hundred terms per row in another order
            torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-6 * top)
