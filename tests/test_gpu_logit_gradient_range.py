"""Logit gradients of ids far below a token's log-sum-exp: probabilities below 2^-126 are values of
bf16 too (down to 2^-133), not zeros."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,v", [(3, 40), (300, 700)])
@pytest.mark.parametrize("every", [1, 7, 150])
def test_probabilities_below_the_smallest_normal(n, v, every):
    """In every token, or in some among others (the waves that have one take another exponential)."""
    from dsv41_rocm import logprob as L

    x = torch.zeros(n, 64, dtype=torch.bfloat16, device="cuda")
    x[:, 0] = 0.125
    x[::every, 0] = 1.0
    w = torch.zeros(v, 64, dtype=torch.bfloat16, device="cuda")
    w[:, 0] = (-80.0 - torch.arange(v, device="cuda") % 13).bfloat16()  # 80 to 92 nats below
    w[0, 0] = 0.0
    t = torch.zeros(n, dtype=torch.int64, device="cuda")
    lse = torch.logsumexp(x.double() @ w.double().t(), 1).float()
    ones = torch.ones(n, device="cuda")
    got = L.logits_grad(x, w, t, 1.0, lse, None, ones, None).double()
    want = -(x.double() @ w.double().t() - lse.double()[:, None]).exp()
    # one bf16 rounding: 2^-8 of normal values, half a step of 2^-133 below them; the fp32 exponent's
    # rounding (z up to 133 binary digits: 2^-17 of z) shows as 2^-16 of the probability
    tol = (2.0 ** -8 + 2.0 ** -16) * want.abs() + 2.0 ** -134
    assert bool(((got - want).abs() <= tol)[:, 1:].all())
    assert bool((got[:, 1:] != 0).all())
