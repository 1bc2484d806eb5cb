"""Arguments of the head gradient's products that are refused before any launch (no GPU needed)."""

import pytest

from dsv41_rocm import _lib


@pytest.mark.parametrize("offset", [4, 8, 12])
def test_dx_refuses_a_misaligned_workspace(offset):
    lib = _lib.load()
    n, v, h = 8, 4096, 64  # cut into ranges, whose sums are stored 16 bytes at a time
    size = lib.dsv41_head_dx_workspace_bytes(n, v, h)
    assert size > 0
    rc = lib.dsv41_head_dx_run(0x1000, v, 0x2000, h, n, v, h, 0x3000, 0, 0x4000 + offset, size, None)
    assert rc == _lib.E_INVALID
    with pytest.raises(ValueError, match="workspace must be 16-byte aligned"):
        _lib.check(rc)
