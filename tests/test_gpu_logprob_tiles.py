"""Fused log-prob and logit gradient at the edges of their tiles: 64-element stages (one to four,
whole and partial), 16-row and 16-token MFMA blocks, the 32-token and 64-row parts of a wave, the
128-row regions and the 256 x 256 tile, against plain 64-bit log-softmax."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [  # tokens, hidden, vocabulary
    (1, 8, 1), (15, 56, 17), (16, 64, 63), (17, 72, 64), (31, 120, 65), (33, 128, 127), (64, 136, 129),
    (97, 184, 191), (127, 192, 255), (129, 200, 256), (160, 256, 257), (255, 64, 385), (257, 72, 511),
    (300, 328, 513), (512, 8, 700), (513, 264, 1025),
]


def _inputs(n, h, v):
    g = torch.Generator(device="cuda").manual_seed(1000 * n + 10 * h + v)
    x = torch.randn(n, h, generator=g, device="cuda").bfloat16()
    w = (0.3 * torch.randn(v, h, generator=g, device="cuda")).bfloat16()
    return x, w, torch.randint(0, v, (n,), generator=g, device="cuda")


def _bound(x, w, temperature):
    """Largest error of a logit summed in 32 bits in any order, over T: h roundings of 2^-24 of
    the sum of the terms' magnitudes; the log-sum-exp and its two log-prob terms double it."""
    mag = float((x.double().abs() @ w.double().abs().t()).max())
    return 2 * (x.shape[1] + 8) * 2.0 ** -24 * mag / temperature + 4e-6


@pytest.mark.parametrize("n,h,v", SHAPES)
def test_forward_tile_edges(n, h, v):
    import dsv41_rocm

    x, w, t = _inputs(n, h, v)
    lp, ent, _ = dsv41_rocm.selected_log_probs(x, w, t, 0.7)
    z = x.double() @ w.double().t() / 0.7
    ref = z.log_softmax(1)
    tol = _bound(x, w, 0.7)
    assert float((lp.double() - ref.gather(1, t[:, None])[:, 0]).abs().max()) <= tol
    # the entropy weighs each logit's error by p |lse - z|, whose sum is at most log v + 1
    want = -(ref.exp() * ref).sum(1)
    assert float((ent.double() - want).abs().max()) <= tol * (2.0 + float(torch.tensor(float(v)).log()))


@pytest.mark.parametrize("n,h,v", SHAPES)
def test_logit_gradient_tile_edges(n, h, v):
    from dsv41_rocm import logprob

    x, w, t = _inputs(n, h, v)
    lse = torch.logsumexp(x.double() @ w.double().t() / 0.7, 1).float()
    g_lp = torch.linspace(-1.0, 1.0, n, device="cuda")
    got = logprob.logits_grad(x, w, t, 0.7, lse, None, g_lp, None)
    z = x.double() @ w.double().t() / 0.7
    p = (z - lse.double()[:, None]).exp()
    want = -g_lp.double()[:, None] * p
    want[torch.arange(n, device="cuda"), t] += g_lp.double()
    want /= 0.7
    # one bf16 rounding, and the probability's relative error from the logit's
    tol = 2.0 ** -8 * want.abs() + 2 * _bound(x, w, 0.7) * g_lp.double().abs()[:, None] / 0.7 * p + 1e-30
    assert bool(((got.double() - want).abs() <= tol).all())
