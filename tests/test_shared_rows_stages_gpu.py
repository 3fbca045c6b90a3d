"""One or two LDS stages (csrc/fa8_shared_rows.h), for one tile of 32 query rows a workgroup and four wavefronts and for two tiles and two wavefronts
each: the stages, and the launches that fill the compute units more than once, are chosen by length and number of the tiles.  Results equal the rolling loop's bit for bit on both sides of each line."""
import ctypes

import pytest
import torch

import cutlass_flash_atten_fp8_amd as fa
from test_shared_rows_gpu import E4, E5, _inputs

pytestmark = pytest.mark.gpu

CASES = [
    # B, H, Hk, Nq, Nk, d, causal, bottom_right, vt, dtype, fp8 out, LDS stages
    (1, 2, 2, 100, 1472, 128, False, False, False, E4, False, 1),   # 23 blocks
    (1, 2, 2, 100, 1473, 128, False, False, False, E4, False, 2),   # 24
    (1, 2, 1, 70, 1600, 64, True, True, True, E5, True, 2),         # v^T
    (1, 2, 2, 97, 3000, 96, True, True, False, E5, False, 2),
    (1, 4, 4, 130, 130, 32, True, False, False, E4, False, 1),
    (1, 3, 3, 200, 190, 64, False, False, False, E4, False, 1),     # 3 blocks: no group is full
    (1, 14, 14, 960, 960, 128, True, False, False, E4, False, 1),   # 420 tiles of unequal length
    (1, 14, 7, 944, 944, 96, True, False, True, E5, True, 1),
    (1, 9, 9, 1990, 1990, 128, True, False, False, E4, False, 1),   # 567 tiles, 32 blocks
    (1, 24, 24, 720, 720, 64, True, False, False, E5, False, 1),    # 552 tiles, 12 blocks
    (1, 20, 20, 1200, 1200, 64, True, False, True, E4, True, 1),    # 760 tiles
    (1, 24, 24, 700, 700, 32, True, False, False, E4, False, 1),
    (1, 24, 12, 700, 1030, 64, False, False, False, E4, False, 1),  # equal tiles, 528 of them, ragged last block
    (2, 12, 12, 992, 1024, 32, False, False, False, E5, True, 1),
    # K and V for one tile or two alone: two stages from fewer blocks on
    (64, 2, 1, 3, 8129, 32, True, True, False, E4, False, 2),       # 64 heads of 128 blocks
    (64, 2, 1, 3, 8100, 32, True, True, False, E4, False, 1),       # of 127
    (16, 64, 64, 1, 1536, 32, False, False, True, E5, True, 2),     # 1024 tiles, 24 blocks
    (1, 24, 24, 90, 43777, 32, True, True, False, E5, False, 2),    # three tiles a head, 685 blocks
    (32, 16, 8, 2, 777, 64, True, True, False, E4, True, 2),        # 256 heads of 13 blocks
    (16, 16, 8, 20, 512, 128, True, True, False, E5, False, 2),     # 128 heads, two tiles each, 8 blocks
    (16, 8, 8, 1, 449, 96, True, True, False, E4, False, 2),
]

TWO_TILES = [
    (1, 56, 56, 519, 519, 64, False, False, False, E4, False, 1),    # 504 workgroups, 9 blocks
    (1, 56, 56, 512, 528, 64, False, False, True, E5, True, 1),      # the same, v^T, a block of 16 keys
    (1, 14, 14, 2432, 2432, 64, False, False, False, E4, False, 2),  # 532, 38 blocks
    (1, 25, 25, 2112, 2112, 64, True, False, True, E5, True, 1),     # 825, more than three a compute unit
    (1, 104, 104, 320, 320, 96, True, False, False, E4, False, 1),   # 520, 5 blocks
    (1, 17, 17, 1600, 1600, 128, True, False, False, E5, False, 2),  # 425, 25 blocks
    (1, 45, 45, 705, 705, 128, False, False, False, E4, False, 1),   # 540, 12 blocks, the last with one key
    (1, 26, 26, 1217, 1232, 128, False, False, True, E5, True, 1),
    (1, 20, 20, 2496, 2496, 96, True, False, True, E4, True, 1),     # 780, 39 blocks
    (1, 32, 32, 1152, 1152, 128, True, False, False, E4, False, 2),  # 576 of unequal length, 18 blocks
    (1, 32, 32, 1094, 1786, 128, True, True, False, E5, False, 1),   # the work of 1.6 a compute unit
    (32, 32, 32, 1, 640, 128, True, True, False, E4, False, 2),      # 1024 heads, 10 blocks
    (32, 32, 32, 2, 576, 96, True, True, True, E5, True, 1),         # 9
    (8, 32, 8, 180, 600, 128, False, False, False, E5, False, 1),    # 768 with the rows of four q heads together: three a compute unit
    (8, 32, 8, 180, 600, 128, True, True, False, E4, False, 1),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}k{}Nq{}Nk{}d{}".format(*c[:6]))
def test_one_tile_a_workgroup_equals_the_rolling_loop_bitwise(case):
    check(case, (32, 4, 1))


@pytest.mark.parametrize("case", TWO_TILES, ids=lambda c: "B{}H{}k{}Nq{}Nk{}d{}c{:d}".format(*c[:7]))
def test_two_tiles_a_workgroup_equal_the_rolling_loop_bitwise(case):
    check(case, (64, 2, 1))


def check(case, plan):
    B, H, Hk, Nq, Nk, d, causal, br, vt, dt, out8, stages = case
    q, k, v = _inputs(Nq + Nk + d, B, H, Hk, Nq, Nk, d, dt)
    v = v.transpose(2, 3).contiguous() if vt else v
    kw = dict(v_transposed=vt, return_lse=True, causal_bottom_right=br, out_dtype=dt if out8 else None)
    want, want_lse = fa.flash_attention_v2_cutlass(q, k, v, causal, d ** -0.5, schedule=fa.FA8_SCHEDULE_ROLLING, **kw)
    got, lse = torch.empty_like(want), torch.empty_like(want_lse)
    p = fa.make_params(q, k, v, got, causal, d ** -0.5, vt, lse, br)
    assert fa.plan(p, with_workspace=False) == plan and fa.form(p, with_workspace=False) == (stages, 1)
    assert fa.lib().fa8_fwd(ctypes.byref(p), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)) and torch.equal(lse, want_lse)
