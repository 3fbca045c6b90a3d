"""Launches of few query rows: two or four wavefronts share 32 of them (csrc/fa8_shared_rows.h).  Every logit, weight and sum is formed
in the same order as by one wavefront, so the result must equal the rolling loop's bit for bit, for every feature of the operator, at
the edges: a single key, a last group of blocks that is not full, row tiles with rows to spare, a workgroup whose second tile is
empty, masks that end inside a block, grouped q heads packed into one tile."""
import pytest
import torch

import cutlass_flash_atten_fp8_amd as fa

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
E4, E5 = torch.float8_e4m3fn, torch.float8_e5m2


def _inputs(seed, B, H, Hk, Nq, Nk, d, dtype):
    g = torch.Generator().manual_seed(seed)
    spread = 3.0 if seed % 2 else 1.0
    return tuple((torch.randn(s, generator=g) * spread).to(dtype).to(DEV) for s in ((B, H, Nq, d), (B, Hk, Nk, d), (B, Hk, Nk, d)))


CASES = [
    # B, H, Hk, Nq, Nk, d, causal, bottom_right, vt, dtype, fp8 out, wavefronts per tile, rows per workgroup
    (1, 1, 1, 1, 1, 128, False, False, False, E4, False, 1, 128),         # a single block is not shared ...
    (1, 2, 2, 33, 64, 64, False, False, False, E4, False, 1, 128),
    (33, 32, 2, 1, 1, 128, False, False, False, E4, False, 2, 64),        # ... unless grouped heads fill the rows
    (40, 32, 1, 2, 48, 256, True, True, True, E5, True, 2, 64),
    (1, 2, 2, 128, 128, 64, True, False, False, E4, True, 4, 32),
    (1, 2, 2, 300, 257, 128, False, False, False, E4, False, 4, 32),      # one key in the second group's first block
    (1, 3, 3, 300, 320, 96, True, True, False, E5, True, 4, 32),
    (1, 2, 2, 700, 100, 128, True, True, False, E4, False, 4, 32),        # queries that see no key
    (1, 2, 1, 200, 336, 160, False, False, True, E4, False, 4, 32),       # v^T, ragged last block
    (2, 6, 2, 5, 777, 192, True, True, False, E4, False, 4, 32),          # 15 packed rows, group of 3
    (1, 16, 2, 9, 1000, 32, True, True, False, E5, False, 4, 32),
    (1, 8, 8, 64, 1023, 224, True, True, False, E4, True, 4, 32),
    (1, 4, 2, 100, 513, 256, True, True, False, E5, True, 4, 32),
    (1, 16, 16, 1024, 1024, 64, True, False, True, E4, True, 4, 32),
    (1, 16, 16, 1024, 1024, 128, True, False, False, E4, False, 4, 64),
    (1, 33, 33, 289, 289, 128, False, False, False, E4, False, 4, 64),    # ten tiles: five workgroups; 330 tiles
    (1, 30, 30, 270, 330, 96, True, True, False, E5, False, 4, 64),       # nine tiles: the last workgroup's second one is empty
    (1, 32, 8, 512, 2000, 128, True, True, False, E4, False, 4, 64),
    (1, 64, 64, 128, 128, 128, False, False, False, E4, False, 4, 32),
    (1, 128, 128, 128, 128, 128, False, False, False, E4, False, 2, 64),  # two blocks only
    (1, 32, 32, 1000, 1000, 128, True, False, False, E4, False, 2, 64),
    (4, 16, 16, 500, 500, 64, False, False, False, E5, False, 2, 64),
    (1, 60, 60, 545, 545, 32, True, False, False, E4, True, 2, 64),       # 18 tiles
    (1, 16, 16, 1056, 1056, 256, True, False, True, E5, True, 2, 64),
    (2, 12, 6, 700, 700, 160, True, False, False, E4, False, 2, 64),
    (40, 64, 16, 3, 130, 128, True, True, False, E4, False, 2, 64),       # 640 k/v heads of one tile (12 rows): no rows in the second tile
    (16, 64, 64, 130, 130, 64, True, False, False, E4, False, 1, 128),    # 5 tiles a head: three pairs for two workgroups, not shared
    (16, 64, 64, 60, 130, 64, True, True, False, E4, False, 2, 64),       # 2 tiles a head: 128-row workgroups would be half idle
    (2, 16, 16, 450, 961, 160, False, False, False, E4, False, 4, 64),    # wide heads, 256 pairs; 16 blocks, the last of one key
    (1, 90, 30, 100, 1500, 192, True, True, False, E5, True, 4, 64),      # 300 packed rows: the last workgroup's second tile is not full
    (1, 14, 14, 1540, 1540, 256, True, False, False, E4, False, 4, 64),   # 350 pairs of unequal length
    (1, 9, 9, 1040, 1040, 224, True, False, True, E5, False, 4, 64),
    (20, 32, 32, 1, 1000, 32, True, True, False, E5, False, 4, 32),       # 640 tiles of one row
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}k{}Nq{}Nk{}d{}".format(*c[:6]) + ("c" if c[6] else "f") + ("vt" if c[8] else ""))
def test_shared_rows_equal_the_rolling_loop_bitwise(case):
    B, H, Hk, Nq, Nk, d, causal, br, vt, dt, out8, waves, rows = case
    q, k, v = _inputs(Nq + Nk + d, B, H, Hk, Nq, Nk, d, dt)
    if vt:
        v = v.transpose(2, 3).contiguous()
    kw = dict(v_transposed=vt, return_lse=True, causal_bottom_right=br, out_dtype=dt if out8 else None)
    want, want_lse = fa.flash_attention_v2_cutlass(q, k, v, causal, d ** -0.5, schedule=fa.FA8_SCHEDULE_ROLLING, **kw)
    got = torch.full(want.shape, float("nan"), dtype=torch.float16, device=DEV).to(want.dtype)
    lse = torch.full_like(want_lse, float("nan"))
    p = fa.make_params(q, k, v, got, causal, d ** -0.5, vt, lse, br)
    assert fa.plan(p, with_workspace=False) == (rows, waves, 1)
    import ctypes
    rc = fa.lib().fa8_fwd(ctypes.byref(p), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, fa.error_string(rc)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
    assert torch.equal(lse, want_lse)


def test_strided_tensors_and_guard_bands():
    """[B,N,H,d] storage (row stride H * d), NaN codes behind the last key, an output whose padding must stay untouched."""
    import ctypes
    B, H, n, d, pad = 2, 3, 200, 128, 72
    kw = {}
    q, k, v = (t.permute(0, 2, 1, 3).contiguous() for t in _inputs(5, B, H, H, n, n, d, E4))

    def spread_out(t):
        buf = torch.full((B, n + pad, H, d), 0x7F, dtype=torch.uint8, device=DEV)
        buf[:, :n] = t.view(torch.uint8)
        return buf.view(E4)[:, :n].permute(0, 2, 1, 3)

    obuf = torch.full((B, n + pad, H, d), 777.0, dtype=torch.float16, device=DEV)
    o = obuf[:, :n].permute(0, 2, 1, 3)
    wide = spread_out(q), spread_out(k), spread_out(v)  # (kept: the parameters hold pointers only)
    p = fa.make_params(*wide, o, False, 0.09, **kw)
    assert fa.plan(p)[1] == 4
    assert fa.lib().fa8_fwd(ctypes.byref(p), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    want = fa.flash_attention_v2_cutlass(*(t.permute(0, 2, 1, 3).contiguous() for t in (q, k, v)), False, 0.09,
                                         schedule=fa.FA8_SCHEDULE_ROLLING)[0]
    torch.cuda.synchronize()
    assert torch.equal(o.contiguous(), want)
    assert (obuf[:, n:] == 777.0).all()


@pytest.mark.parametrize("shape", [(1, 4, 2, 40, 700, 64), (1, 16, 16, 256, 700, 128), (1, 40, 40, 700, 700, 64), (1, 8, 8, 300, 700, 256)],
                         ids=lambda s: "B{}H{}k{}Nq{}Nk{}d{}".format(*s))
@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("code", [0x7C, 0x7F], ids=["inf", "nan"])  # of e5m2
def test_infinity_and_nan_reach_the_rows_that_they_reach_in_the_rolling_loop(shape, where, code):
    """One element of one head, full attention.  An infinite key gives a row a logit of +inf (NaN row), or of -inf (the key is not seen)."""
    q, k, v = _inputs(2, *shape, E5)
    t = {"q": q, "k": k, "v": v}[where]
    t.view(torch.uint8)[0, 1, 33 if where == "q" else 432, 17] = code
    outs = []
    for schedule in (fa.FA8_SCHEDULE_ROLLING, fa.FA8_SCHEDULE_AUTO):
        outs += fa.flash_attention_v2_cutlass(q, k, v, False, 0.125, return_lse=True, schedule=schedule)
    want, want_lse, got, lse = outs
    assert fa.plan(fa.make_params(q, k, v, got, False, 0.125, lse=lse))[1:] in ((2, 1), (4, 1))
    torch.cuda.synchronize()
    assert not torch.isfinite(want).all() and torch.isfinite(want).any()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got[~torch.isnan(got)], want[~torch.isnan(want)])
    assert torch.equal(torch.isnan(lse), torch.isnan(want_lse)) and torch.equal(lse[~torch.isnan(lse)], want_lse[~torch.isnan(want_lse)])


def test_one_block_of_a_wide_head_is_not_shared():
    for n, waves in ((64, 1), (65, 2)):
        q, k, v = _inputs(n, 1, 4, 4, n, n, 160, E4)
        o = torch.empty(q.shape, dtype=torch.float16, device=DEV)
        assert fa.plan(fa.make_params(q, k, v, o, False, 0.08))[1] == waves
