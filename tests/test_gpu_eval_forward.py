"""An eval-mode forward leaves the curvature evaluations out: the outputs that
it returns and the generator's state are those of the full evaluation."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grad_type", ["finite_difference", "analytic"])
def test_eval_forward_equals_the_training_forward(dev, grad_type):
    from angelo_amd import scenes
    from test_gpu_pipeline import _field_model
    model = _field_model(dev, grad_type=grad_type)
    rays, _ = scenes.config0_batch(n_rays=300, n_views=4, seed=5)
    rays = rays.to(dev)
    samples = scenes.uniform_samples(rays, 33)
    states, outs = [], []
    for training in (True, False):
        model.train(training)
        torch.manual_seed(3)
        with torch.no_grad():
            outs.append(model.forward_(rays, samples))
        states.append(torch.cuda.get_rng_state())
    assert torch.equal(*states)
    for k in outs[1]:
        assert torch.equal(outs[0][k], outs[1][k]), k
    assert "sdf_laplace_samples" in outs[0] and "sdf_laplace_samples" not in outs[1]
