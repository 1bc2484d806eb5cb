"""Batches on both sides of the rules of csrc/slice_rule.h, with histories longer than a slice's
tables of small ones: ids, kept sets and statuses exactly the oracle's, log-probs within 1e-4."""

import pytest
import torch

from test_gpu_sampler_small import DEV, _agrees, _batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,vocab,history", [(3, 40003, 2101), (3, 40003, 5100), (3, 40003, 5200), (40, 20001, 900),
                                                (40, 20001, 2700)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("knobs", [{"top_p": 0.9}, {"min_p": 0.02}])
def test_top_p_and_min_p(rows, vocab, history, dtype, knobs):
    full, u, hist = _batch(rows, vocab, dtype, rows + history, history)
    _agrees(full, vocab, u, hist, temperature=0.8, repetition_penalty=1.1, frequency_penalty=0.1, **knobs)


@pytest.mark.parametrize("rows,vocab,history", [(260, 20001, 1000), (260, 20001, 1100), (5, 33001, 4000), (100, 33001, 4000)])
def test_full_vocabulary_and_replay(rows, vocab, history):
    import dsv41_rocm

    full, u, hist = _batch(rows, vocab, torch.bfloat16, rows + history, history)
    _agrees(full, vocab, u, hist, temperature=0.7, presence_penalty=0.4)
    logits, h = full.to(DEV)[:, :vocab], hist.to(DEV)
    r = dsv41_rocm.sample(logits, uniforms=u.to(DEV), history=h, temperature=0.7, presence_penalty=0.4)
    again = dsv41_rocm.replay_log_probs(logits, r.ids, history=h, temperature=0.7, presence_penalty=0.4)
    assert torch.equal(again, r.logprobs)
