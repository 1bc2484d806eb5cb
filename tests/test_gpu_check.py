"""The check behind a launch (dsv41_check_wait): set statuses and ids outside their range are seen
wherever they lie, from every thread and stream, and a call after a failed one starts clean."""

import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1025, 4096, 4097, 70001, 300001])
def test_check_finds_any_status_and_any_id(n):
    from dsv41_rocm._check import any_set

    status = torch.zeros(n, dtype=torch.int32, device="cuda")
    ids = torch.randint(0, 50, (n,), device="cuda")
    assert any_set(status, ids, 50) == (False, False)
    for at in {0, n // 2, n - 1}:
        status[at] = 1 << 30
        assert any_set(status) == (True, False)
        status[at] = 0
        for bad in (-1, 50, 1 << 40):
            kept = ids[at].clone()
            ids[at] = bad
            assert any_set(None, ids, 50) == (False, True)
            assert any_set(status, ids, 50) == (False, True)
            ids[at] = kept
    assert any_set(status, ids, 50) == (False, False)
    assert any_set(status[:0], ids[:0], 50) == (False, False)


def test_check_from_threads_and_streams():
    from dsv41_rocm._check import any_set

    wrong = []

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            status = torch.zeros(1000, dtype=torch.int32, device="cuda")
            if k % 2:
                status[k] = 4
            for _ in range(50):
                if any_set(status) != (bool(k % 2), False):
                    wrong.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_scoring_refuses_ids_outside_the_vocabulary():
    import dsv41_rocm

    x = torch.randn(70, 64, device="cuda").bfloat16()
    w = torch.randn(300, 64, device="cuda").bfloat16()
    t = torch.randint(0, 300, (70,), device="cuda")
    good = dsv41_rocm.selected_log_probs(x, w, t)[0]
    for bad in (-1, 300):
        u = t.clone()
        u[69] = bad
        for kw in ({}, {"check": False}):
            with pytest.raises(ValueError, match="target token ID is outside the model vocabulary"):
                dsv41_rocm.selected_log_probs(x, w, u, **kw)
    assert torch.equal(dsv41_rocm.selected_log_probs(x, w, t)[0], good)
    mask = torch.zeros(7, 10, dtype=torch.bool, device="cuda")
    mask[2:5, 3:] = True
    lp = dsv41_rocm.token_log_probs(x.view(7, 10, 64), w, t.view(7, 10), mask, 1.0)
    assert torch.equal(lp[mask], good.view(7, 10)[mask]) and not lp[~mask].any()
