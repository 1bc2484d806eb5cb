"""Small top-p and min-p batches cut into slices (small_*_kernel), full-vocabulary batches spread
over the GPU beyond 128 rows, and vector loads over rows that end inside a vector: ids, kept sets
and statuses exactly the oracle's, log-probs within 1e-4, at the edges of their ranges."""

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


PENALTIES = [(0, {}), (40, {"repetition_penalty": 1.2}), (300, {"presence_penalty": 0.4, "frequency_penalty": 0.3}),
             (77, {"repetition_penalty": 0.7, "presence_penalty": -0.5})]


@pytest.mark.parametrize("rows,vocab", [(1, 18433), (3, 20011), (17, 24577), (128, 18500), (129, 18500), (2, 151851)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("history,pen", PENALTIES)
def test_top_p_slices(rows, vocab, dtype, history, pen):
    for i, top_p in enumerate((0.9, 0.01, 0.9995)):
        full, u, hist = _batch(rows, vocab, dtype, 7 * rows + i, history)
        _agrees(full, vocab, u, hist, temperature=(0.8, 1.0, 0.6)[i], top_p=top_p, **pen)
    _agrees(full, vocab, u, hist, temperature=0.8, top_p=0.9, greedy=True, **pen)


@pytest.mark.parametrize("rows,vocab", [(1, 18433), (3, 20011), (200, 18500), (256, 18500), (257, 18500), (2, 151851)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("history,pen", PENALTIES)
def test_min_p_slices(rows, vocab, dtype, history, pen):
    for i, knobs in enumerate(({"min_p": 0.05}, {"min_p": 0.3, "top_p": 0.8}, {"min_p": 0.001})):
        full, u, hist = _batch(rows, vocab, dtype, 11 * rows + i, history)
        _agrees(full, vocab, u, hist, temperature=(0.8, 1.0, 0.6)[i], **knobs, **pen)
    _agrees(full, vocab, u, hist, temperature=0.8, min_p=0.05, greedy=True, **pen)


@pytest.mark.parametrize("knobs", [{"top_p": 0.9}, {"min_p": 0.05}])
def test_slices_of_odd_rows(knobs):
    """Flat rows (more tokens at the boundary than the lists hold: the fallback), one far token, a
    NaN, an infinity, the type's lowest value, a bad uniform and a bad history id."""
    V = 20011
    full, u, hist = _batch(9, V, torch.float32, 5, 30)
    full[0, :V] = 0.25
    full[1, :V] = -50.0
    full[1, 15000] = 50.0
    full[2, 19999] = float("nan")
    full[3, 3] = float("inf")
    full[4, 77] = float("-inf")
    full[5, :V:3] = torch.finfo(torch.float32).min
    u[6] = 1.5
    hist[7, 5] = V
    full[8, :V] = torch.round(full[8, :V])  # many ties
    _agrees(full, V, u, hist, temperature=1.0, repetition_penalty=1.1, **knobs)
    _agrees(full, V, u, None, temperature=0.7, **knobs)


@pytest.mark.parametrize("rows", [128, 129, 256, 257, 300, 448, 449])
@pytest.mark.parametrize("history,pen", PENALTIES[:3])
def test_spread_full_vocabulary(rows, history, pen):
    import dsv41_rocm

    V = 9001
    full, u, hist = _batch(rows, V, torch.bfloat16, rows, history)
    _agrees(full, V, u, hist, temperature=0.7, **pen)
    logits, h = full.to(DEV)[:, :V], None if hist is None else hist.to(DEV)
    r = dsv41_rocm.sample(logits, uniforms=u.to(DEV), history=h, temperature=0.7, **pen)
    again = dsv41_rocm.replay_log_probs(logits, r.ids, history=h, temperature=0.7, **pen)
    assert torch.equal(again, r.logprobs)  # bit for bit, whichever way either was cut


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
