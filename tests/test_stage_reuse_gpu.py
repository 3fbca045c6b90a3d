"""A K or V stage is overwritten only when every wavefront's reads of it have returned, also by copies of blocks that do not exist, which write their zeros
at once: many short workgroups side by side, whose stores and LDS traffic delay each other's reads; every launch must give the same bits."""
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
