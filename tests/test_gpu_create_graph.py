"""Gradients of the scoring head under create_graph, whichever operands require them: the values of
a plain backward, and an error (not a missing term) where they are differentiated again."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _score(op, x, w, t):
    import dsv41_rocm

    if op:
        return torch.ops.dsv41_rocm.selected_log_probs(x, w, t, 0.9, None, 2.0)[:2]
    return dsv41_rocm.selected_log_probs(x, w, t, 0.9)[:2]


# which operands require a gradient, and which gradients are asked for
CASES = [("xw", "x"), ("xw", "w"), ("x", "x"), ("w", "w")]


@pytest.mark.parametrize("op", [False, True])
@pytest.mark.parametrize("n", [0, 5, 200])
@pytest.mark.parametrize("have,ask", CASES)
@pytest.mark.parametrize("loss", ["linear", "square"])
def test_second_derivatives_raise(op, n, have, ask, loss):
    g = torch.Generator(device="cuda").manual_seed(n + 1)
    x = torch.randn(n, 64, generator=g, device="cuda").bfloat16().requires_grad_("x" in have)
    w = torch.randn(300, 64, generator=g, device="cuda").bfloat16().requires_grad_("w" in have)
    t = torch.randint(0, 300, (n,), generator=g, device="cuda")
    leaf = {"x": x, "w": w}[ask]

    def total():
        lp, ent = _score(op, x, w, t)
        return (lp + ent).sum() if loss == "linear" else (lp * lp + ent).sum()

    try:
        (first,) = torch.autograd.grad(total(), leaf, create_graph=True)
    except RuntimeError:  # (refused at once where both require gradients)
        assert have == "xw"
        return
    assert torch.equal(first, torch.autograd.grad(total(), leaf)[0])
    with pytest.raises(RuntimeError, match="cannot be differentiated again"):
        first.float().pow(2).sum().backward()


@pytest.mark.parametrize("op", [False, True])
def test_a_penalty_on_the_gradient_is_not_left_out(op):
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(9, 64, generator=g, device="cuda").bfloat16().requires_grad_()
    w = torch.randn(300, 64, generator=g, device="cuda").bfloat16()
    t = torch.randint(0, 300, (9,), generator=g, device="cuda")
    lp = _score(op, x, w, t)[0]
    (dx,) = torch.autograd.grad(lp.sum(), x, create_graph=True)
    with pytest.raises(RuntimeError):
        (lp.sum() + dx.float().pow(2).sum()).backward()
