"""The old and behavior vectors of the losses carry no derivative of any kind into them."""

import pytest
import torch
import torch.autograd.forward_ad as fwad

from dsv41_rocm.tis import _vector


def test_vectors_are_detached_from_both_kinds_of_derivatives():
    like = torch.zeros(3)
    plain = torch.tensor([-1.0, -2.0, -0.5])
    with fwad.dual_level():
        for value in (plain, plain.double(), plain.clone().requires_grad_(), [-1.0, -2.0, -0.5],
                      fwad.make_dual(plain, torch.ones(3)), fwad.make_dual(plain.clone().requires_grad_(), torch.ones(3))):
            got = _vector(value, like)
            assert got.dtype == torch.float32 and not got.requires_grad
            assert fwad.unpack_dual(got).tangent is None
            assert torch.equal(got, plain)


@pytest.mark.gpu
def test_losses_take_vectors_with_tangents():
    import dsv41_rocm as d

    g = torch.Generator(device="cuda").manual_seed(2)
    new = lambda: [-torch.rand(4 + i, generator=g, device="cuda") for i in range(3)]
    cur, old, beh, adv = [p.requires_grad_() for p in new()], new(), new(), [1.0, -0.5, 0.25]
    calls = (lambda o, b: d.decoupled_token_tis_loss(cur, o, b, adv)[0], lambda o, b: d.grpo_loss(cur, b, adv)[0],
             lambda o, b: d.grpo_loss(cur, b, adv, 0.2, o, 0.1)[0])
    for call in calls:
        want = call(old, beh)
        with fwad.dual_level():
            dual = lambda ts: [fwad.make_dual(t, torch.ones_like(t)) for t in ts]
            got = call(dual(old), dual(beh))
            assert torch.equal(got, want)
            grads = torch.autograd.grad(got, cur)
        assert all(torch.equal(a, b) for a, b in zip(grads, torch.autograd.grad(want, cur)))
