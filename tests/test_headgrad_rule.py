"""Which dw of the scoring backward takes the hand-written kernel: where it was timed faster than the
library GEMM, whatever the count of tokens (no GPU needed)."""

import pytest

from dsv41_rocm.logprob import _own_dw

# tokens, vocabulary columns, hidden; hand-written / library as timed
CASES = [
    (300, 129280, 7168, True),  # 0.86: a ragged count, as most are
    (100, 129280, 7168, True),  # 0.93
    (500, 64000, 4608, True),  # 0.85
    (256, 129280, 7168, False),  # 1.13
    (128, 151936, 2048, False),  # 1.06
    (256, 151936, 2048, True),  # 0.90
    (150, 151936, 2048, True),  # 0.80
    (1000, 129280, 7168, True),  # 0.89
    (2048, 2000, 7168, True),  # 0.87, 224 tiles
    (128, 25600, 512, True),  # 0.76
    (300, 16000, 512, True),  # 0.88, 126 tiles
    (2048, 16000, 512, False),  # 1.30
    (16384, 1000, 512, False),  # 3.05
    (64, 151936, 2048, False),  # (few tokens: the library's throughout)
]


@pytest.mark.parametrize("n,columns,h,own", CASES)
def test_dw_goes_where_it_is_faster(n, columns, h, own):
    assert _own_dw(n, columns, h) is own
