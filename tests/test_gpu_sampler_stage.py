"""Slices of small top-p and min-p batches that collect as many tokens as their LDS stage holds, one
fewer and more, and rows whose lists just fill and overflow: exactly the oracle's draws."""

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def _agrees(logits, u, **knobs):
    import dsv41_rocm

    got = dsv41_rocm.sample(logits.cuda(), uniforms=u.cuda(), **knobs)
    ids, lps, kept, status = oracle.sample(logits.float().numpy(), uniforms=u.numpy(), **knobs)
    assert not status.any()
    assert np.array_equal(got.ids.cpu().numpy(), ids)
    assert np.array_equal(got.kept.cpu().numpy(), kept)
    assert np.max(np.abs(got.logprobs.cpu().numpy() - lps)) <= 1e-4


@pytest.mark.parametrize("rows,vocab", [(1, 20011), (100, 20011), (16, 151936)])
@pytest.mark.parametrize("count", [1, 1023, 1024, 1025, 2049, 4095, 4096, 4097, 9000])
@pytest.mark.parametrize("spread", [False, True])
@pytest.mark.parametrize("knobs", [{"top_p": 0.9}, {"min_p": 0.05}])
def test_lists_at_the_stage_and_row_limits(rows, vocab, count, spread, knobs):
    """``count`` tokens at one value (top-p: the boundary's; min-p: within the bound), in a row or
    spread over all slices, beside one that is likelier and a far tail."""
    logits = torch.full((rows, vocab), -30.0)
    first = 4000
    at = torch.arange(count) * ((vocab - first) // count) if spread else torch.arange(count)
    for r in range(rows):
        logits[r, first - r + at] = 0.0
    # the likely token holds half of the mass (top-p), or stands one above (min-p)
    logits[:, 7] = float(np.log(count)) if "top_p" in knobs else 1.0
    u = torch.rand(rows, generator=torch.Generator().manual_seed(count))
    _agrees(logits, u, **knobs)
