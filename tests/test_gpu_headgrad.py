"""The two products of the head's backward (dsv41_head_dx_run, dsv41_head_dw_run) at the edges of
their tiles: 64-deep stages of the contraction (whole and partial), 256 x 256 tiles, 8-element chunks,
contraction ranges, accumulation over vocabulary ranges, against 64-bit products of the operands."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [  # tokens, vocabulary, hidden
    (1, 1, 8), (7, 63, 16), (16, 64, 64), (33, 65, 72), (64, 129, 128), (65, 257, 136), (127, 300, 248),
    (128, 511, 256), (200, 1000, 264), (257, 513, 520), (300, 4099, 200), (513, 777, 1024), (70, 20011, 512),
]


def _close(got, want, mag, k):
    """bf16 rounding of an fp32 sum of k products: 2^-9 of the result and k 2^-24 of the terms."""
    tol = 2.0 ** -8 * want.abs() + (k + 8) * 2.0 ** -24 * mag + 1e-30
    return bool(((got.double() - want).abs() <= tol).all())


def _lib():
    from dsv41_rocm import _lib as m

    return m, m.load(), torch.cuda.current_stream().cuda_stream


def _operands(n, v, h):
    g0 = torch.Generator(device="cuda").manual_seed(n + 3 * v + 7 * h)
    gs = (v + 7) // 8 * 8 + 8
    g = torch.full((n, gs), float("nan"), device="cuda").bfloat16()
    g[:, :(v + 7) // 8 * 8] = 0
    g[:, :v] = torch.randn(n, v, generator=g0, device="cuda")
    w = torch.randn(v, h + 8, generator=g0, device="cuda").bfloat16()[:, :h]
    x = torch.randn(n, h + 16, generator=g0, device="cuda").bfloat16()[:, :h]
    return g, w, x


@pytest.mark.parametrize("n,v,h", SHAPES)
def test_dx_tile_edges(n, v, h):
    m, lib, stream = _lib()
    g, w, _ = _operands(n, v, h)
    want = g[:, :v].double() @ w.double()
    mag = g[:, :v].double().abs() @ w.double().abs()
    ws_bytes = lib.dsv41_head_dx_workspace_bytes(n, v, h)
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device="cuda")
    args = (g.data_ptr(), g.stride(0), w.data_ptr(), w.stride(0), n, v, h)
    dx = torch.full((n, h), float("nan"), device="cuda").bfloat16()
    m.check(lib.dsv41_head_dx_run(*args, dx.data_ptr(), 0, ws.data_ptr(), ws_bytes, stream))
    assert _close(dx, want, mag, v)
    acc = torch.full((n, h), float("nan"), device="cuda")
    m.check(lib.dsv41_head_dx_run(*args, acc.data_ptr(), 1, None, 0, stream))
    assert bool(((acc.double() - want).abs() <= (v + 8) * 2.0 ** -24 * mag + 1e-30).all())
    m.check(lib.dsv41_head_dx_run(*args, acc.data_ptr(), 2, None, 0, stream))
    assert bool(((acc.double() - 2 * want).abs() <= 3 * (v + 8) * 2.0 ** -24 * mag + 1e-30).all())
    if ws_bytes:
        assert lib.dsv41_head_dx_run(*args, dx.data_ptr(), 0, None, 0, stream) == m.E_WORKSPACE


@pytest.mark.parametrize("n,v,h", SHAPES)
def test_dw_tile_edges(n, v, h):
    m, lib, stream = _lib()
    g, _, x = _operands(n, v, h)
    dw = torch.full((v, h + 8), 3.0, device="cuda").bfloat16()
    m.check(lib.dsv41_head_dw_run(g.data_ptr(), g.stride(0), x.data_ptr(), x.stride(0), n, v, h, dw.data_ptr(),
                                  dw.stride(0), stream))
    want = g[:, :v].double().t() @ x.double()
    mag = g[:, :v].double().abs().t() @ x.double().abs()
    assert _close(dw[:, :h], want, mag, n)
    assert bool((dw[:, h:] == 3.0).all())


def test_gradients_over_vocabulary_ranges():
    from dsv41_rocm import logprob

    n, v, h = 300, 3001, 264
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(n, h, generator=gen, device="cuda").bfloat16()
    w = (0.2 * torch.randn(v, h, generator=gen, device="cuda")).bfloat16()
    t = torch.randint(0, v, (n,), generator=gen, device="cuda")
    lse = torch.logsumexp(x.double() @ w.double().t(), 1).float()
    g_lp = torch.randn(n, generator=gen, device="cuda")
    one = logprob.selected_log_probs_backward(x, w, t, 1.0, lse, None, g_lp, None)
    for chunk in (256, 777, 1500):
        many = logprob.selected_log_probs_backward(x, w, t, 1.0, lse, None, g_lp, None, vocab_chunk=chunk)
        for a, b in zip(one, many):
            assert float((a.double() - b.double()).norm()) <= 4e-3 * float(a.double().norm())
    empty = logprob.selected_log_probs_backward(x[:0], w, t[:0], 1.0, lse[:0], None, g_lp[:0], None)
    assert empty[0].shape == (0, h) and not empty[1].any()


def test_refused_before_launch():
    m, lib, stream = _lib()
    g, w, x = _operands(8, 64, 64)
    for bad in ((g.data_ptr(), 63), (g.data_ptr() + 2, g.stride(0))):
        assert lib.dsv41_head_dx_run(*bad, w.data_ptr(), w.stride(0), 8, 64, 64, x.data_ptr(), 0, None, 0, stream) < 0
        assert lib.dsv41_head_dw_run(*bad, x.data_ptr(), x.stride(0), 8, 64, 64, w.data_ptr(), 72, stream) < 0
    assert lib.dsv41_head_dx_run(g.data_ptr(), g.stride(0), w.data_ptr(), w.stride(0), 8, 64, 60, x.data_ptr(), 0, None,
                                 0, stream) == m.E_UNSUPPORTED


def test_vocabulary_above_the_offset_limit():
    """A head whose whole row of logit gradients would pass the products' 32-bit block offsets."""
    from dsv41_rocm.logprob import MAX_GRAD_COLUMNS, selected_log_probs

    n, v, h = 3, 2 * MAX_GRAD_COLUMNS + 9, 8
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(n, h, generator=g, device="cuda").bfloat16().requires_grad_()
    w = torch.randn(v, h, generator=g, device="cuda").bfloat16().requires_grad_()
    t = torch.tensor([0, MAX_GRAD_COLUMNS, v - 1], device="cuda")
    selected_log_probs(x, w, t)[0].sum().backward()
    x64, w64 = (p.detach().double().requires_grad_() for p in (x, w))
    torch.log_softmax(x64 @ w64.t(), -1).gather(1, t[:, None]).sum().backward()
    # bf16 logit gradients and results: 2^-8 of the terms' magnitudes, which one term and the mean
    # of the rows under the softmax (at most 1 by weight) make up
    mag = w64.detach().abs()[t] + w64.detach().abs().max()
    assert bool(((x.grad.double() - x64.grad).abs() <= 2.0 ** -7 * mag).all())
    assert bool(((w.grad[t].double() - w64.grad[t]).abs() <= 2.0 ** -7 * (w64.grad[t].abs() + x64.detach().abs().sum(0))).all())


@pytest.mark.parametrize("n", [0, 5, 100])
def test_second_derivatives_are_refused(n):
    """The kernels record no graph, on either side of the token count that picks them."""
    from dsv41_rocm.logprob import selected_log_probs

    x = torch.randn(n, 64, device="cuda").bfloat16().requires_grad_()
    w = torch.randn(300, 64, device="cuda").bfloat16().requires_grad_()
    lp = selected_log_probs(x, w, torch.zeros(n, dtype=torch.int64, device="cuda"))[0]
    with pytest.raises(RuntimeError):
        torch.autograd.grad(lp.sum(), (x, w), create_graph=True)
    assert all(torch.isfinite(g).all() for g in torch.autograd.grad(
        selected_log_probs(x, w, torch.zeros(n, dtype=torch.int64, device="cuda"))[0].sum(), (x, w)))
