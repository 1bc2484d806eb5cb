"""What lies in a row's padding changes neither what a batch draws nor how long it takes.  (The
vector loads of an odd bf16 row read one element of it.)"""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _time(fn):
    best = float("inf")
    for _ in range(12):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        fn()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


@pytest.mark.parametrize("rows,knobs", [(300, {"top_k": 50}), (1024, {"top_k": 50}), (1024, {"top_k": 200}),
                                        (300, {"top_k": 300, "min_p": 0.01})])
def test_padding_of_odd_rows_sends_none_to_a_second_look(rows, knobs):
    """A second look at a row reads it again by single loads: 2.0 to 2.6 times the time."""
    import dsv41_rocm

    vocab = 151851
    g = torch.Generator(device="cuda").manual_seed(rows)
    full = torch.zeros(rows, 151936, dtype=torch.bfloat16, device="cuda")
    full[:, :vocab] = 2 * torch.randn(rows, vocab, generator=g, device="cuda")
    u = torch.rand(rows, generator=g, device="cuda")
    call = lambda: dsv41_rocm.sample(full[:, :vocab], uniforms=u, check=False, **knobs)
    want, plain = call(), _time(call)
    for pad in (float("-inf"), float("inf"), float("nan"), -3.0e38):
        full[:, vocab:] = pad
        got = call()
        assert torch.equal(got.ids, want.ids) and torch.equal(got.kept, want.kept) and not got.status.any()
        assert torch.equal(got.logprobs, want.logprobs)
        assert _time(call) < 1.5 * plain
