"""A K or V stage is overwritten only when every wavefront's reads of it have returned, also by copies of blocks that do not exist, which write their zeros
at once: many short workgroups side by side, whose stores and LDS traffic delay each other's reads; every launch must give the same bits."""
import ctypes

import pytest
import torch

import cutlass_flash_atten_fp8_amd as fa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 130, 200, 320])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
def test_every_launch_of_every_loop_gives_the_same_bits(n, d, causal):
    g = torch.Generator(device="cuda").manual_seed(n)
    q, k, v = ((torch.randn((16, 64, n, d), device="cuda", generator=g)).to(torch.float8_e4m3fn) for _ in range(3))
    want = fa.flash_attention_v2_cutlass(q, k, v, causal, d ** -0.5, schedule=fa.FA8_SCHEDULE_ROLLING)[0]
    for schedule in (fa.FA8_SCHEDULE_ROLLING, fa.FA8_SCHEDULE_PIPELINED, fa.FA8_SCHEDULE_DENSE):
        for _ in range(6):
            assert torch.equal(fa.flash_attention_v2_cutlass(q, k, v, causal, d ** -0.5, schedule=schedule)[0], want), schedule


@pytest.mark.parametrize("shape", [(16, 64, 64, 32), (16, 64, 200, 32), (16, 64, 320, 96), (8, 32, 130, 256), (8, 32, 320, 192), (1, 64, 4096, 128)],
                         ids=lambda s: "B{}H{}N{}d{}".format(*s))
@pytest.mark.parametrize("vt", [False, True], ids=["rows", "vt"])
@pytest.mark.parametrize("dt", [torch.float8_e4m3fn, torch.float8_e5m2], ids=["e4m3", "e5m2"])
def test_every_launch_of_the_other_loops_gives_the_same_bits(shape, vt, dt):
    """Half a copy pass a tile (head dim 32), the rolling loop of head dims without others, two stages (above 128); many heads of long sequences."""
    B, H, n, d = shape
    n = n // 16 * 16 if vt else n
    g = torch.Generator(device="cuda").manual_seed(n)
    q, k, v = ((torch.randn((B, H, n, d), device="cuda", generator=g)).to(dt) for _ in range(3))
    v = v.transpose(2, 3).contiguous() if vt else v
    want = fa.flash_attention_v2_cutlass(q, k, v, True, d ** -0.5, v_transposed=vt, schedule=fa.FA8_SCHEDULE_ROLLING)[0]
    for _ in range(6):
        for schedule in (fa.FA8_SCHEDULE_ROLLING, fa.FA8_SCHEDULE_PIPELINED):
            assert torch.equal(fa.flash_attention_v2_cutlass(q, k, v, True, d ** -0.5, v_transposed=vt, schedule=schedule)[0], want)


@pytest.mark.parametrize("shape", [(1, 16, 16, 1024, 1024, 64), (1, 8, 8, 900, 2000, 32), (1, 8, 4, 300, 1100, 96), (1, 3, 3, 500, 1300, 128),  # one tile a workgroup
                                   (1, 32, 8, 512, 2056, 128), (1, 30, 30, 320, 1376, 96),                                                   # two, four wavefronts
                                   (1, 30, 30, 1504, 1536, 32), (1, 20, 20, 2080, 2112, 64), (1, 20, 20, 1600, 1632, 128)],
                         ids=lambda s: "B{}H{}k{}Nq{}Nk{}d{}".format(*s))
@pytest.mark.parametrize("vt", [False, True], ids=["rows", "vt"])
def test_every_launch_with_sums_apart_gives_the_same_bits(shape, vt):
    B, H, Hk, nq, nk, d = shape
    nk = nk // 16 * 16 if vt else nk
    g = torch.Generator(device="cuda").manual_seed(nk)
    q, k, v = (torch.randn((B, h, n, d), device="cuda", generator=g).to(torch.float8_e4m3fn) for h, n in ((H, nq), (Hk, nk), (Hk, nk)))
    v = v.transpose(2, 3).contiguous() if vt else v
    call = lambda: fa.flash_attention_v2_cutlass(q, k, v, True, d ** -0.5, v_transposed=vt, causal_bottom_right=True)[0]
    want = call()
    assert fa.lib().fa8_fwd_apart(ctypes.byref(fa.make_params(q, k, v, want, True, d ** -0.5, vt, causal_bottom_right=True))) == 1
    for _ in range(12):
        assert torch.equal(call(), want)
