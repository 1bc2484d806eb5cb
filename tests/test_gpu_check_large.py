"""The check behind a launch over many values: set statuses and ids outside their range are seen at
every position around the 16-byte groups' edges and on either side of the size that is left to
tensor operations, from any alignment, and it takes no longer than those."""

import time

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 5, 4095, 4099, 16384 + 7, 65536 + 5])
@pytest.mark.parametrize("skip", [0, 1, 2, 3])
def test_every_position_from_every_alignment(n, skip):
    from dsv41_rocm._check import any_set

    status = torch.zeros(n + 8, dtype=torch.int32, device="cuda")[skip:skip + n]
    ids = torch.zeros(n + 8, dtype=torch.int64, device="cuda")[skip:skip + n]
    status._base[skip + n:] = 1  # (behind the last value)
    ids._base[skip + n:] = -1
    status._base[:skip] = 1
    ids._base[:skip] = 50
    assert any_set(status, ids, 50) == (False, False)
    places = sorted({p % n for p in (0, 1, 2, 3, 4, n // 2, n - 5, n - 4, n - 3, n - 2, n - 1, 4096, 16383, 16384)})
    for p in places:
        status[p] = 2
        assert any_set(status, ids, 50) == (True, False)
        status[p] = 0
        for bad in (50, -1, -(1 << 62)):
            ids[p] = bad
            assert any_set(status, ids, 50) == (False, True)
        ids[p] = 49
    assert any_set(None, ids, 0)[1] and any_set(None, ids, -3)[1]


@pytest.mark.parametrize("n", [1 << 18, (1 << 18) + 1, 3_000_000])
def test_sizes_left_to_tensor_operations(n):
    from dsv41_rocm._check import any_set

    status = torch.zeros(n, dtype=torch.int32, device="cuda")
    ids = torch.zeros(n, dtype=torch.int64, device="cuda")
    assert any_set(status) == (False, False) and any_set(status, ids, 1) == (False, False)
    status[n - 1], ids[n - 2] = 4, 1
    assert any_set(status) == (True, False) and any_set(None, ids, 1) == (False, True)
    assert any_set(status, ids, 1) == (True, True)


@pytest.mark.parametrize("n", [500_000, 1_000_000, 4_000_000])
def test_no_slower_than_tensor_operations(n):
    """(One load in flight per thread took 2.1, 3.9 and 36 times as long.)"""
    from dsv41_rocm._check import any_set

    def best(fn):
        fn()
        times = []
        for _ in range(30):
            torch.cuda.synchronize()
            t = time.perf_counter()
            fn()
            times.append(time.perf_counter() - t)
        return min(times)

    status = torch.zeros(n, dtype=torch.int32, device="cuda")
    assert best(lambda: any_set(status)) <= 1.5 * best(lambda: bool((status != 0).any()))
