"""Fused log-prob and logit gradient at the edges of their tiles: 64-element stages (one to four,
whole and partial), 16-row and 16-token MFMA blocks, the 32-token and 64-row parts of a wave, the
128-row regions and the 256 x 256 tile, and on each way of cutting a call into workgroups,
against plain 64-bit log-softmax."""

import math

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
    assert float((ent.double() - want).abs().max()) <= tol * (2.0 + math.log(v))


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


# the other cuts of a call into workgroups: the 512 x 128 tile (three blocks of tokens; one, with
# the vocabulary shared evenly by rows), even row ranges of the 256 x 256 one, and two runs of
# token blocks with ranges of their own (64 blocks of four ranges, the 65th of 129; 256 blocks of one
# range, the other two of 12).  test_logprob_cuts.py asserts that each takes its cut.
ROUTES = [(331, 64, 40003), (100, 1024, 131071), (200, 1024, 60011), (16390, 128, 33001), (66000, 8, 3000)]


@pytest.mark.parametrize("n,h,v", ROUTES)
def test_cuts_of_large_heads(n, h, v):
    import dsv41_rocm
    from dsv41_rocm import logprob

    x, w, t = _inputs(n, h, v)
    w = (w.float() * 0.1).bfloat16()
    lp, ent, _ = dsv41_rocm.selected_log_probs(x, w, t, 0.7)
    lse = torch.empty(n, device="cuda")
    g_lp = torch.linspace(-1.0, 1.0, n, device="cuda")
    spans = [(b, min(n, b + 2048)) for b in range(0, n, 2048)]
    for b, e in spans:
        z = x[b:e].double() @ w.double().t() / 0.7
        ref = z.log_softmax(1)
        tol = _bound(x[b:e], w, 0.7)
        assert float((lp[b:e].double() - ref.gather(1, t[b:e, None])[:, 0]).abs().max()) <= tol
        assert float((ent[b:e].double() + (ref.exp() * ref).sum(1)).abs().max()) <= tol * (2.0 + math.log(v))
        lse[b:e] = torch.logsumexp(z, 1)
    got = logprob.logits_grad(x, w, t, 0.7, lse, None, g_lp, None)
    for b, e in spans:
        g = g_lp[b:e].double()[:, None]
        p = (x[b:e].double() @ w.double().t() / 0.7 - lse[b:e].double()[:, None]).exp()
        want = -g * p
        want[torch.arange(e - b, device="cuda"), t[b:e]] += g[:, 0]
        want /= 0.7
        tol = 2.0 ** -8 * want.abs() + 2 * _bound(x[b:e], w, 0.7) * g.abs() / 0.7 * p + 1e-30
        assert bool(((got[b:e].double() - want).abs() <= tol).all())
