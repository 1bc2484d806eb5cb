"""dx in contraction ranges of its own: each way of writing it (bf16, fp32, onto fp32), with the
workspace and without, over tile counts that fill a round of CUs, just pass it, and leave most idle,
against 64-bit products of the operands."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# tokens, vocabulary, hidden: 1, 2, 4 and 9 tiles; 144 (three ranges in two rounds); 256 and 289
# tiles; ranges of unequal stages, and a last one that is partial
SHAPES = [(5, 1024, 8), (200, 4099, 264), (300, 1030, 512), (520, 2111, 520), (2100, 9001, 4104), (2048, 2000, 8192),
          (4100, 3003, 4104)]


@pytest.mark.parametrize("n,v,h", SHAPES)
def test_dx_of_every_mode(n, v, h):
    from dsv41_rocm import _lib as m

    lib, stream = m.load(), torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device="cuda").manual_seed(n + v)
    gs = (v + 7) // 8 * 8
    g = torch.zeros(n, gs, dtype=torch.bfloat16, device="cuda")
    g[:, :v] = torch.randn(n, v, generator=gen, device="cuda")
    w = torch.randn(v, h, generator=gen, device="cuda").bfloat16()
    want = g[:, :v].double() @ w.double()
    mag = g[:, :v].double().abs() @ w.double().abs()
    tol = (v + 8) * 2.0 ** -24 * mag + 1e-30  # v roundings of an fp32 sum in any order
    size = lib.dsv41_head_dx_workspace_bytes(n, v, h)
    args = (g.data_ptr(), gs, w.data_ptr(), h, n, v, h)
    for space in ((size, 0) if size else (0,)):
        ws = torch.full((max(space, 16),), 0xFF, dtype=torch.uint8, device="cuda")  # (NaNs)
        ptr = ws.data_ptr() if space else None
        out = torch.full((n, h), float("nan"), device="cuda")
        m.check(lib.dsv41_head_dx_run(*args, out.data_ptr(), 1, ptr, space, stream))
        assert bool(((out.double() - want).abs() <= tol).all())
        before = out.double()
        m.check(lib.dsv41_head_dx_run(*args, out.data_ptr(), 2, ptr, space, stream))
        assert bool(((out.double() - before - want).abs() <= tol + 2.0 ** -23 * out.double().abs()).all())
        if space or not size:
            low = torch.full((n, h), float("nan"), device="cuda").bfloat16()
            m.check(lib.dsv41_head_dx_run(*args, low.data_ptr(), 0, ptr, space, stream))
            assert bool(((low.double() - want).abs() <= 2.0 ** -8 * want.abs() + tol).all())
