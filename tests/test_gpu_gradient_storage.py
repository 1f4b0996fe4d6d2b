"""Gradients of autograd.render: the lights' lie in memory of their own, apart from the materials'."""
import pytest

from eos_amd import scenes

pytestmark = pytest.mark.gpu


def test_light_gradients_hold_their_own_memory():
    import torch
    from eos_amd import _lib as E, autograd as G
    s = scenes.config_a(32, 32)
    g = E.Scene(s)
    params = [p.requires_grad_() for p in G.params_of(s)]
    grads = torch.autograd.grad(G.render(g, *params).sum(), params)
    materials, lights = grads[:3], grads[3:]
    assert all(x.shape == p.shape for x, p in zip(grads, params))
    kept = {x.untyped_storage().data_ptr(): x.untyped_storage().nbytes() for x in lights}
    assert not {x.untyped_storage().data_ptr() for x in materials} & set(kept)
    assert all(n == 4 * 6 * len(s.lights) for n in kept.values())
