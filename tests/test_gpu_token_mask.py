"""token_log_probs over masks of any rank, a single token's among them."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(), (1,), (7,), (1, 1), (3, 5), (2, 3, 4), (0, 4)])
@pytest.mark.parametrize("fill", [True, False, None])
def test_masks_of_any_rank(shape, fill):
    import dsv41_rocm

    g = torch.Generator(device="cuda").manual_seed(len(shape))
    hidden = torch.randn(*shape, 64, generator=g, device="cuda").bfloat16()
    w = torch.randn(300, 64, generator=g, device="cuda").bfloat16()
    t = torch.randint(0, 300, shape, generator=g, device="cuda")
    mask = torch.rand(shape, generator=g, device="cuda") < 0.5 if fill is None else torch.full(shape, fill, device="cuda")
    got = dsv41_rocm.token_log_probs(hidden, w, t, mask, 0.8)
    want = torch.zeros(shape, device="cuda")
    if bool(mask.any()):
        lp = dsv41_rocm.score_targets(hidden[mask], w, t[mask], 0.8)
        want = want.masked_scatter(mask, lp)
    assert got.shape == want.shape and torch.equal(got, want)
