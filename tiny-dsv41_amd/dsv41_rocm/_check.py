"""Whether a launch left a status bit set, or was given an id outside its range: one native call
that launches a one-workgroup check and watches a word of pinned memory for its answer (tensor
operations for hundreds of thousands of values)."""

from __future__ import annotations

import threading
from typing import Optional

import torch

from . import _lib


class _Word(threading.local):
    """A thread's word, made at its first use (pinned memory needs a GPU).  The call that uses it
    returns only with the answer, so a thread never has two in flight, whatever streams and
    devices it uses."""

    ptr = None

    def make(self):
        self.host = torch.zeros(1, dtype=torch.int32, device="cpu", pin_memory=True)
        self.ptr = self.host.data_ptr()


_word = _Word()
# More statuses or ids than these are reduced by tensor operations over the whole GPU, with the host's
# wait behind them.  combine_states, whose check finds its statuses in no cache, takes 179 us for
# 500000 tokens with the one-workgroup check and 177 with tensor operations, for 1000000 323 and 301,
# for 100000 61 and 81.
MAX_VALUES = 1 << 18

_left: list = []  # words of calls that failed: their launch may still write them


def any_set(status: Optional[torch.Tensor], ids: Optional[torch.Tensor] = None, limit: int = 0) -> tuple[bool, bool]:
    """(some status is nonzero, some id lies outside [0, limit)) of contiguous int32 statuses and
    int64 ids on one GPU, after everything queued on its current stream."""
    t = status if status is not None else ids
    n = status.numel() if status is not None else 0
    n_ids = ids.numel() if ids is not None else 0
    if n == 0 and n_ids == 0:
        return False, False
    if max(n, n_ids) > MAX_VALUES:
        return n > 0 and bool((status != 0).any()), n_ids > 0 and bool(((ids < 0) | (ids >= limit)).any())
    if _word.ptr is None:
        _word.make()
    device = t.device
    with torch.cuda.device(device):
        got = _lib.load().dsv41_check_wait(status.data_ptr() if n else None, n, ids.data_ptr() if n_ids else None,
                                           n_ids, limit, _word.ptr, torch.cuda.current_stream(device).cuda_stream)
    if got < 0:
        _left.append(_word.host)
        _word.make()
        _lib.check(got)
    return bool(got & 1), bool(got & 2)
