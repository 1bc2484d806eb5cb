"""Vector loads over rows that end inside a vector: ids, kept sets and statuses exactly the
oracle's, log-probs within 1e-4, whatever lies behind the rows."""

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _batch(rows, vocab, dtype, seed, history=0, pad=None, scale=2.0):
    """Logits as a view of padded rows whose padding is NaN and inf, uniforms and history."""
    g = torch.Generator().manual_seed(seed)
    stride = (vocab + 15) // 8 * 8 if pad is None else vocab + pad
    full = torch.full((rows, stride), float("nan"), dtype=dtype)
    full[:, 1::2] = float("inf")
    full[:, :vocab] = (scale * torch.randn(rows, vocab, generator=g)).to(dtype)
    hist = torch.randint(-3, vocab, (rows, history), generator=g) if history else None
    if hist is not None:  # likely tokens among them, some more than once
        top = full[:, :vocab].float().topk(min(8, vocab), 1).indices
        hist[:, : min(history, top.shape[1])] = top[:, : min(history, top.shape[1])]
        hist[:, -1] = top[:, 0]
    return full, torch.rand(rows, generator=g), hist


def _agrees(full, vocab, u, hist, **knobs):
    import dsv41_rocm

    logits = full.to(DEV)[:, :vocab]
    got = dsv41_rocm.sample(logits, uniforms=u.to(DEV), history=None if hist is None else hist.to(DEV), check=False,
                            **knobs)
    ids, lps, kept, status = oracle.sample(full[:, :vocab].float().numpy(), uniforms=u.numpy(),
                                           history=None if hist is None else hist.numpy(), **knobs)
    assert np.array_equal(got.status.cpu().numpy(), status)
    assert np.array_equal(got.ids.cpu().numpy(), ids)
    assert np.array_equal(got.kept.cpu().numpy(), kept)
    fine = status == 0
    assert np.max(np.abs(got.logprobs.cpu().numpy()[fine] - lps[fine]), initial=0.0) <= 1e-4


@pytest.mark.parametrize("vocab", [255, 1001, 4095, 4098, 9003, 151851])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("knobs", [{}, {"top_k": 20}, {"top_k": 20, "min_p": 0.05}, {"top_k": 300, "top_p": 0.9},
                                   {"top_p": 0.9}, {"min_p": 0.05}, {"top_k": 3000, "top_p": 0.95}])
def test_rows_ending_inside_a_vector(vocab, dtype, knobs):
    full, u, hist = _batch(3, vocab, dtype, vocab, 20)
    _agrees(full, vocab, u, None, temperature=0.7, **knobs)
    _agrees(full, vocab, u, hist, temperature=1.0, repetition_penalty=1.2, **knobs)
    vocab = min(vocab, 5001)
    full, u, _ = _batch(270, vocab, dtype, vocab + 1)
    _agrees(full, vocab, u, None, temperature=0.7, **knobs)
