"""The checked calls and the losses under a default device other than the CPU (``torch.device`` as
a context, ``torch.set_default_device``): the same answers.  Each case runs in a thread of its own,
whose first checked call makes the thread's pinned word."""

import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

V, N, H = 900, 12, 64


def _inputs():
    g = torch.Generator(device="cuda").manual_seed(3)
    logits = torch.randn(N, V, generator=g, device="cuda")
    u = torch.rand(N, generator=g, device="cuda")
    x = torch.randn(N, H, generator=g, device="cuda").bfloat16()
    w = torch.randn(V, H, generator=g, device="cuda").bfloat16()
    t = torch.randint(0, V, (N,), generator=g, device="cuda")
    lps = [-torch.rand(5 + i, generator=g, device="cuda") for i in range(3)]
    return logits, u, x, w, t, lps, torch.tensor([1.0, -0.5, 0.25], device="cpu")


def _calls():
    import dsv41_rocm as d

    logits, u, x, w, t, lps, adv = _inputs()
    half = V // 2
    grid = torch.ones(3, 4, dtype=torch.bool, device="cuda")

    def merged():
        shards = [d.sample_shard(logits[:, b:e], vocab_offset=b, vocab_size=V, top_k=20) for b, e in ((0, half), (half, V))]
        return d.merge_shards(shards, top_k=20, uniforms=u).ids

    def full_shards():
        parts = [(logits[:, b:e], b) for b, e in ((0, half), (half, V))]
        states = [d.full_shard_states(z, vocab_offset=b, vocab_size=V) for z, b in parts]
        masses = [d.full_shard_masses(z, states, shard_index=i, vocab_offset=b, vocab_size=V) for i, (z, b) in enumerate(parts)]
        picks = [d.full_shard_draw(z, states, masses, shard_index=i, vocab_offset=b, vocab_size=V, uniforms=u)
                 for i, (z, b) in enumerate(parts)]
        return d.full_shard_finish(states, picks, vocab_size=V, uniforms=u).ids

    return {
        "sample": lambda: d.sample(logits, uniforms=u, top_k=20).ids,
        "replay": lambda: d.replay_log_probs(logits, t),
        "merge_shards": merged,
        "full_shards": full_shards,
        "selected_log_probs": lambda: d.selected_log_probs(x, w, t)[0],
        "unchecked": lambda: d.selected_log_probs(x, w, t, check=False)[0],
        "score_targets": lambda: d.score_targets(x, w, t, 0.8),
        "token_log_probs": lambda: d.token_log_probs(x.view(3, 4, H), w, t.view(3, 4), grid, 0.8),
        "combine_states": lambda: d.combine_states(d.shard_states(x, w, t, 0.8, 0)[None])[0],
        "tis": lambda: d.decoupled_token_tis_loss(lps, lps, lps, adv)[0],
        "grpo": lambda: d.grpo_loss(lps, lps, adv)[0],
    }


@pytest.mark.parametrize("name", ["sample", "replay", "merge_shards", "full_shards", "selected_log_probs", "unchecked",
                                  "score_targets", "token_log_probs", "combine_states", "tis", "grpo"])
def test_default_device(name):
    want = _calls()[name]()
    got = []

    def work():
        with torch.device("cuda"):
            try:
                got.append(_calls()[name]())
            except Exception as e:  # noqa: BLE001
                got.append(e)

    t = threading.Thread(target=work)
    t.start()
    t.join()
    assert isinstance(got[0], torch.Tensor), got[0]
    assert torch.equal(got[0], want)
