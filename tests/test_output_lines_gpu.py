"""O leaves the kernels in pieces of 4 - 8 bytes a lane where few rows are written, and as whole lines through LDS where many are (whole_lines in the library).
Same bits: heads of a call with lines are also run by themselves, in pieces.  Every head dim and both output types, a last tile that is not full, rows of O that are 8-byte
aligned only and apart, with guard bands; query counts on both sides of the line."""
import ctypes

import pytest
import torch

import cutlass_flash_atten_fp8_amd as fa

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
E4, E5 = torch.float8_e4m3fn, torch.float8_e5m2


def _call(q, k, v, o, causal, lse, rows_schedule):
    p = fa.make_params(q, k, v, o, causal, q.shape[3] ** -0.5, False, lse)
    p.schedule = fa.FA8_SCHEDULE_ROLLING if rows_schedule else fa.FA8_SCHEDULE_AUTO
    assert fa.lib().fa8_fwd(ctypes.byref(p), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0


@pytest.mark.parametrize("d", [32, 64, 96, 128, 160, 192, 224, 256])
@pytest.mark.parametrize("out8", [False, True], ids=["fp16", "fp8"])
@pytest.mark.parametrize("heads,n,shared", [(180, 330, False), (24, 150, False), (513, 33, False), (600, 32, False), (33, 250, True), (33, 248, True), (20, 900, True)],
                         ids=lambda x: str(x))
def test_lines_and_pieces_give_the_same_bits(d, out8, heads, n, shared):
    g = torch.Generator().manual_seed(d + n)
    dt = E5 if n % 2 else E4
    q, k, v = ((torch.randn((1, heads, n, d), generator=g) * 1.5).to(dt).to(DEV) for _ in range(3))
    out = dt if out8 else torch.float16
    pad = 8 if out8 else 4  # elements: rows that are 8-byte aligned only
    buf = torch.zeros((1, n + 3, heads, d + pad), dtype=torch.float16, device=DEV).fill_(3.0).to(out)
    before = buf.clone()
    o = buf[:, :n, :, :d].permute(0, 2, 1, 3)
    lse = torch.empty((1, heads, n), dtype=torch.float32, device=DEV)
    _call(q, k, v, o, True, lse, not shared)
    for at in range(0, heads, 1 + heads // 15):  # at most 1.4 MB of O, in the rolling loop: pieces
        few = slice(at, min(heads, at + 3))
        part = torch.empty((1, few.stop - at, n, d), dtype=out, device=DEV)
        part_lse = torch.empty((1, few.stop - at, n), dtype=torch.float32, device=DEV)
        _call(q[:, few].contiguous(), k[:, few].contiguous(), v[:, few].contiguous(), part, True, part_lse, True)
        assert torch.equal(o[:, few].contiguous().view(torch.uint8), part.view(torch.uint8)), at
        assert torch.equal(lse[:, few], part_lse)
    before[:, :n, :, :d] = buf[:, :n, :, :d]
    assert torch.equal(buf.view(torch.uint8), before.view(torch.uint8))  # nothing but the rows was written
