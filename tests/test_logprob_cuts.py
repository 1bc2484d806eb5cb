"""The cut that each route of test_gpu_logprob_tiles.py is there for, read from the workspace it
asks for (one 16-byte state for every vocabulary range of every token; no GPU needed)."""

import ctypes

import pytest

from dsv41_rocm import _lib
from test_gpu_logprob_tiles import ROUTES

STATES = {
    (331, 64, 40003): 331 * 79,  # 79 blocks of 512 rows (157 of 256): the tall tile
    (100, 1024, 131071): 100 * 256,  # a range for every CU
    (200, 1024, 60011): 200 * 256,  # more ranges than the 235 blocks of 256 rows: cut by rows
    (16390, 128, 33001): 16384 * 4 + 6 * 129,  # two runs: 64 token blocks, and the 65th
    (66000, 8, 3000): 65536 + 464 * 12,  # two runs: 256 token blocks of one range, and two more of 12
}


@pytest.mark.parametrize("route", ROUTES)
def test_routes_take_their_cut(route):
    n, h, v = route
    d = _lib.LogprobDesc()
    d.struct_size = ctypes.sizeof(_lib.LogprobDesc)
    d.n_tokens, d.hidden, d.vocab = n, h, v
    d.x = d.w = d.targets = d.out_logprob = 0x1000
    d.x_row_stride = d.w_row_stride = h
    d.temperature = 1.0
    assert _lib.load().dsv41_logprob_workspace_bytes(ctypes.byref(d)) == 16 * STATES[route]
