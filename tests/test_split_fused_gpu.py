"""Split keys in one kernel (fa8_split_fused_kernel): workgroups take the row max of those before them from the workspace.  What the other tests
of split keys do not reach: a workgroup that stops waiting and forms that max itself, workspaces with the state of earlier calls, several
streams, ranges of every length up to the two-kernel form."""
import ctypes

import pytest
import torch

import cutlass_flash_atten_fp8_amd as fa
from test_split_kv_gpu import DEV, E4, E5, _inputs, assert_same_up_to_sum_order

pytestmark = pytest.mark.gpu

# B, H, Hk, Nq, Nk, d, causal, vt, dtype
CASES = [
    (1, 8, 2, 1, 6001, 128, True, False, E4),
    (1, 6, 2, 2, 8191, 96, True, False, E5),
    (1, 8, 1, 5, 7777, 128, True, False, E4),    # two row tiles, the second with 8 rows
    (1, 8, 2, 1, 8192, 32, True, False, E5),
    (1, 4, 4, 3, 4112, 160, False, True, E4),    # v^T, ragged last block
    (1, 8, 2, 1, 20000, 256, True, False, E4),
    (1, 4, 2, 50, 12345, 64, True, False, E4),   # masks in several blocks, four tiles
]


def call(q, k, v, o, causal, vt=False, lse=None, late=0):
    """One call through fa8_fwd_ws_late on a workspace of the size asked for."""
    p = fa.make_params(q, k, v, o, causal, q.shape[3] ** -0.5, vt, lse, True)
    assert fa.plan(p)[2] > 1 and fa.form(p) == (0, 1)
    need = ctypes.c_int64()
    assert fa.lib().fa8_fwd_workspace(ctypes.byref(p), ctypes.byref(need)) == 0
    ws = torch.empty(need.value, dtype=torch.uint8, device=DEV)
    rc = fa.lib().fa8_fwd_ws_late(ctypes.byref(p), ws.data_ptr(), need.value, late, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, fa.error_string(rc)
    torch.cuda.synchronize()


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}k{}Nq{}Nk{}d{}".format(*c[:6]))
def test_a_workgroup_that_does_not_wait_forms_the_maximum_itself(case):
    """No workgroup hands on its maximum, or the first, the second, the last but one or every other one does not: the same bits."""
    B, H, Hk, Nq, Nk, d, causal, vt, dt = case
    q, k, v = _inputs(Nk + d, B, H, Hk, Nq, Nk, d, dt)
    k.view(torch.uint8)[0, 0, 70, 3] = 0x7C if dt == E5 else 0x7E  # infinity, the largest finite number
    v = v.transpose(2, 3).contiguous() if vt else v
    want, want_lse = fa.flash_attention_v2_cutlass(q, k, v, causal, d ** -0.5, v_transposed=vt, return_lse=True, causal_bottom_right=True)
    splits = fa.plan(fa.make_params(q, k, v, want, causal, d ** -0.5, vt, want_lse, True))[2]
    for late in (0, 0xFFFFFFFF, 1, 2, 1 << splits - 2, 0x55555555):
        got, lse = torch.full_like(want, float("nan")), torch.full_like(want_lse, float("nan"))
        call(q, k, v, got, causal, vt, lse, late)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)) and torch.equal(lse.view(torch.int32), want_lse.view(torch.int32))


def test_one_late_part_costs_its_own_keys_alone():
    """16 blocks a wavefront in 32 parts: with one maximum late a workgroup reads the keys of that part again, not those of all before it."""
    q, k, v = _inputs(1, 1, 8, 2, 1, 131072, 128, E4)
    o = torch.empty(q.shape, dtype=torch.float16, device=DEV)

    def microseconds(late):
        times = []
        for _ in range(5):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            call(q, k, v, o, True, late=late)
            end.record()
            torch.cuda.synchronize()
            times.append(begin.elapsed_time(end) * 1e3)
        return sorted(times)[2]
    one, all_of_them = microseconds(1), microseconds(0xFFFFFFFF)
    assert 2 * one < all_of_them, (one, all_of_them)


def test_a_workspace_with_the_state_of_earlier_calls():
    """The same workspace for calls with other keys, other lengths, other splits: no value of an earlier call is taken."""
    ws = torch.zeros(64 << 20, dtype=torch.uint8, device=DEV)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for seed, nk in enumerate((8000, 8000, 5000, 16000, 8000)):
        q, k, v = _inputs(seed, 1, 8, 2, 1, nk, 128, E4)
        if seed % 2 == 0:
            k = (k.float() * 0.25).to(E4)
        o = torch.full(q.shape, float("nan"), dtype=torch.float16, device=DEV)
        p = fa.make_params(q, k, v, o, True, 0.09, causal_bottom_right=True)
        need = ctypes.c_int64()
        assert fa.form(p) == (0, 1)
        assert fa.lib().fa8_fwd_workspace(ctypes.byref(p), ctypes.byref(need)) == 0 and 0 < need.value <= ws.numel()
        assert fa.lib().fa8_fwd_ws(ctypes.byref(p), ws.data_ptr(), need.value, stream) == 0
        torch.cuda.synchronize()
        assert torch.equal(o, fa.flash_attention_v2_cutlass(q, k, v, True, 0.09, causal_bottom_right=True)[0])


@pytest.mark.parametrize("group", [1, 4, 8, 16, 32])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_ranges_of_many_lengths(d, group):
    """One to fifteen blocks a wavefront, in one kernel and, where the logits of many rows do not fit in LDS, in two."""
    for nk in (4096, 9000, 30011, 120001):
        q, k, v = _inputs(nk + group, 1, group, 1, 1, nk, d, E4)
        if 2 * nk * d > 40e6:
            continue
        want = fa.flash_attention_v2_cutlass(q, k, v, True, d ** -0.5, causal_bottom_right=True, schedule=fa.FA8_SCHEDULE_ROLLING)[0]
        got = fa.flash_attention_v2_cutlass(q, k, v, True, d ** -0.5, causal_bottom_right=True)[0]
        torch.cuda.synchronize()
        assert fa.plan(fa.make_params(q, k, v, got, True, d ** -0.5, causal_bottom_right=True))[2] > 1
        assert_same_up_to_sum_order(got, want, v, nk)


# the blocks of a wavefront whose logits just fit in LDS, for head dim and rows
@pytest.mark.parametrize("d,rows,fit", [(32, 16, 8), (64, 8, 15), (96, 16, 5), (128, 4, 23), (160, 8, 3), (256, 4, 7)])
def test_the_longest_ranges_of_one_kernel(d, rows, fit):
    """32 parts of four ranges that are all as long as fits, the last one a key shorter, and one block more, which takes two kernels."""
    for nk, kernels in ((32 * 4 * fit * 64 - 1, 1), (32 * 4 * fit * 64 + 1, 2)):
        q, k, v = _inputs(nk + rows, 1, rows, 1, 1, nk, d, E4)
        want = fa.flash_attention_v2_cutlass(q, k, v, True, d ** -0.5, causal_bottom_right=True, schedule=fa.FA8_SCHEDULE_ROLLING)[0]
        got = fa.flash_attention_v2_cutlass(q, k, v, True, d ** -0.5, causal_bottom_right=True)[0]
        torch.cuda.synchronize()
        p = fa.make_params(q, k, v, got, True, d ** -0.5, causal_bottom_right=True)
        assert fa.plan(p)[2] > 1 and fa.form(p) == (0, kernels)
        assert_same_up_to_sum_order(got, want, v, nk)


def test_two_streams():
    """Calls side by side on two streams, each with more workgroups than half the compute units."""
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    ins = [_inputs(i, 2, 32, 8, 1, 20000, 128, E4) for i in range(2)]
    want = [fa.flash_attention_v2_cutlass(*t, True, 0.09, causal_bottom_right=True)[0] for t in ins]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(10):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i].append(fa.flash_attention_v2_cutlass(*ins[i], True, 0.09, causal_bottom_right=True)[0])
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(o, want[i]) for o in got[i])
