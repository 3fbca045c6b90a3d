"""Wavefronts that share 32 query rows and keep the sums of their own KV blocks apart (fa8_shared_rows_kernel with APART, through fa8_fwd_any_order, which
the bindings call).  Weights are those of the rolling loop bit for bit, the fp32 sums over the keys are taken in another order.  Both sides of
the lines of the rule; groups that are not full (fewer blocks than wavefronts in the last), one key in the last block, workgroups whose second tile is empty or not
full, masks that end inside a block, queries that see no key, packed rows of grouped q heads, both layouts of v, all formats."""
import ctypes

import pytest
import torch

import cutlass_flash_atten_fp8_amd as fa
from oracle import fa8_oracle as fo
from oracle.parity_gate import assert_parity
from test_parity_gpu import sample_rows
from test_split_kv_gpu import DEV, E4, E5, _inputs, assert_same_up_to_sum_order

pytestmark = pytest.mark.gpu

CASES = [
    # B, H, Hk, Nq, Nk, d, causal, bottom_right, vt, dtype, fp8 out, (rows per workgroup, wavefronts per tile), sums apart
    (1, 2, 2, 100, 704, 64, False, False, False, E4, False, (32, 4), False),     # 11 blocks
    (1, 2, 2, 100, 705, 64, False, False, False, E4, False, (32, 4), True),      # 12, the last with one key
    (1, 4, 2, 70, 784, 64, True, True, True, E5, False, (32, 4), True),           # 13 blocks: one in the last group; v^T, ragged
    (1, 8, 8, 1200, 800, 64, True, True, False, E4, False, (32, 4), True),       # queries that see no key
    (1, 16, 16, 1024, 1024, 64, True, False, False, E4, False, (32, 4), True),   # two tiles a compute unit
    (1, 16, 16, 1024, 1024, 64, True, False, False, E4, True, (32, 4), False),   # fp8 output: the bits of fa8_fwd
    (2, 6, 2, 11, 900, 32, True, True, False, E4, False, (32, 4), True),         # 33 packed rows, group of 3
    (1, 4, 4, 90, 1030, 32, False, False, False, E5, False, (32, 4), True),
    (1, 8, 4, 40, 1100, 96, True, True, False, E4, False, (32, 4), True),
    (1, 2, 2, 40, 1100, 96, False, False, False, E5, False, (32, 4), True),
    (1, 3, 3, 200, 1216, 128, True, False, True, E4, False, (32, 4), False),     # 19 blocks
    (1, 3, 3, 200, 1232, 128, False, False, True, E4, False, (32, 4), True),      # 20
    (1, 8, 8, 32, 1300, 128, False, False, False, E4, False, (32, 4), False),    # one tile a k/v head
    (1, 16, 4, 512, 3001, 128, True, True, False, E4, False, (32, 4), True),
    (1, 32, 32, 500, 760, 96, False, False, False, E4, False, (64, 4), True),    # 12 blocks
    (1, 30, 30, 290, 1330, 96, True, True, False, E5, False, (64, 4), True),      # ten tiles
    (1, 30, 30, 270, 1330, 128, True, True, False, E4, False, (64, 4), True),    # nine: the last workgroup's second one is empty
    (1, 32, 8, 512, 2000, 128, True, True, False, E4, False, (64, 4), True),
    (1, 11, 11, 1400, 1408, 128, False, False, True, E5, False, (64, 4), True),
    (1, 24, 24, 1300, 1300, 64, False, False, False, E4, False, (64, 2), True),  # two tiles, two wavefronts each; 21 blocks
    (1, 20, 20, 2100, 2100, 64, True, False, False, E4, False, (64, 2), True),    # 33 blocks, 660 pairs of unequal length
    (1, 30, 30, 1500, 1504, 32, False, False, True, E5, False, (64, 2), True),
    (1, 28, 28, 1100, 1100, 96, True, False, False, E4, False, (64, 2), True),
    (1, 45, 45, 705, 705, 96, False, False, False, E4, False, (64, 2), False),   # 540 pairs; two a compute unit run at once
    (3, 30, 10, 250, 2101, 128, False, False, False, E4, False, (64, 2), True),  # instead of unshared rows
    (1, 20, 20, 1600, 1600, 128, True, False, False, E5, False, (64, 2), True),   # 25 blocks
    # tiles of unequal length, more pairs than the first line lets through: both sides of blocks and of pairs a compute unit
    (1, 40, 40, 1536, 1536, 32, True, False, False, E4, False, (64, 2), True),    # 24 blocks, 960 pairs
    (1, 40, 40, 1472, 1472, 32, True, False, False, E4, False, (64, 2), False),   # 23
    (1, 86, 86, 1536, 1536, 32, True, False, False, E4, False, (64, 2), False),   # 2064 pairs: more than eight
    (1, 20, 20, 3072, 3072, 64, True, False, True, E4, False, (64, 2), True),     # 48, 960
    (1, 20, 20, 3008, 3008, 64, True, False, False, E4, False, (64, 2), False),   # 47
    (1, 27, 27, 3072, 3072, 64, True, False, False, E4, False, (64, 2), False),   # 1296: more than five
    (1, 12, 12, 3072, 3072, 96, True, False, False, E5, False, (64, 2), True),    # 48, 576
    (1, 12, 12, 3008, 3008, 96, True, False, False, E4, False, (64, 2), False),   # 47
    (1, 12, 12, 3072, 3072, 128, True, False, True, E4, False, (64, 2), True),
    (1, 12, 12, 3008, 3008, 128, True, False, False, E4, False, (64, 2), False),
    (1, 17, 17, 3072, 3072, 128, True, False, False, E4, False, (64, 2), False),  # 816: more than three
    # one tile a workgroup, two to three of them a compute unit
    (1, 20, 20, 1056, 1056, 32, False, False, False, E4, False, (32, 4), True),   # 660 tiles
    (1, 7, 7, 3072, 3072, 64, False, False, False, E4, False, (32, 4), True),     # 672, 48 blocks
    (1, 7, 7, 3008, 3008, 64, False, False, True, E5, False, (32, 4), False),     # 47
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}k{}Nq{}Nk{}d{}".format(*c[:6]) + ("c" if c[6] else "f") + ("vt" if c[8] else ""))
def test_sums_apart_against_the_rolling_loop(case):
    B, H, Hk, Nq, Nk, d, causal, br, vt, dt, out8, cut, apart = case
    q, k, v = _inputs(Nq + Nk + d, B, H, Hk, Nq, Nk, d, dt)
    if vt:
        v = v.transpose(2, 3).contiguous()
    kw = dict(v_transposed=vt, return_lse=True, causal_bottom_right=br, out_dtype=dt if out8 else None)
    want, want_lse = fa.flash_attention_v2_cutlass(q, k, v, causal, d ** -0.5, schedule=fa.FA8_SCHEDULE_ROLLING, **kw)
    p = fa.make_params(q, k, v, want, causal, d ** -0.5, vt, want_lse, br)
    assert fa.lib().fa8_fwd_apart(ctypes.byref(p)) == apart
    if fa.plan(p, fa.FA8_PLAN_ANY_ORDER)[0] != 128 or apart:
        assert fa.plan(p, fa.FA8_PLAN_ANY_ORDER) == cut + (1,)
    got, lse = fa.load_extension().flash_attention_v2_cutlass(q, k, v, causal, d ** -0.5, **kw)
    again, lse2 = torch.full_like(want, float("nan")), torch.full_like(want_lse, float("nan"))
    p = fa.make_params(q, k, v, again, causal, d ** -0.5, vt, lse2, br)
    assert fa.lib().fa8_fwd_any_order(ctypes.byref(p), None, 0, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.uint8), again.view(torch.uint8)) and torch.equal(lse, lse2)
    empty = torch.isneginf(want_lse)
    assert torch.equal(torch.isneginf(lse), empty) and (got.float()[empty] == 0).all()
    assert_same_up_to_sum_order(got, want, v, Nk)
    assert (lse - want_lse)[~empty].abs().max() <= 5e-6 * max(1.0, want_lse[~empty].abs().max().item())
    if not apart:
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
    # without leave to reorder, the same bits as the rolling loop
    plain = torch.empty_like(want)
    p.o = plain.data_ptr()
    assert fa.lib().fa8_fwd_ws(ctypes.byref(p), None, 0, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    assert torch.equal(plain.view(torch.uint8), want.view(torch.uint8))


@pytest.mark.parametrize("shape", [(1, 4, 2, 40, 1300, 64), (1, 16, 16, 300, 1300, 128), (1, 16, 16, 1024, 1400, 96)], ids=lambda s: "B{}H{}k{}Nq{}Nk{}d{}".format(*s))
@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("code", [0x7C, 0x7F], ids=["inf", "nan"])  # of e5m2
def test_infinity_and_nan_reach_the_rows_that_they_reach_in_the_rolling_loop(shape, where, code):
    """One element of one head, full attention.  An infinite key gives a row a logit of +inf (NaN row), or of -inf (the key is not seen)."""
    q, k, v = _inputs(2, *shape, E5)
    t = {"q": q, "k": k, "v": v}[where]
    t.view(torch.uint8)[0, 1, 33 if where == "q" else 632, 17] = code
    outs = []
    for schedule in (fa.FA8_SCHEDULE_ROLLING, fa.FA8_SCHEDULE_AUTO):
        outs += fa.flash_attention_v2_cutlass(q, k, v, False, 0.125, return_lse=True, schedule=schedule)
    want, want_lse, got, lse = outs
    assert fa.lib().fa8_fwd_apart(ctypes.byref(fa.make_params(q, k, v, got, False, 0.125, lse=lse))) == 1
    torch.cuda.synchronize()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    assert not torch.isfinite(want).all() and torch.isfinite(want).any()
    fine = torch.isfinite(want)
    v = v.float()
    assert_same_up_to_sum_order(got[fine], want[fine], torch.where(torch.isfinite(v), v, torch.zeros_like(v)), shape[4])
    assert torch.equal(torch.isnan(lse), torch.isnan(want_lse))
    seen = ~torch.isnan(want_lse)
    assert (lse - want_lse)[seen].abs().max() <= 5e-6 * max(1.0, want_lse[seen].abs().max().item())


@pytest.mark.parametrize("vt", [False, True], ids=["rows", "vt"])
def test_strided_tensors_and_guard_bands(vt):
    """[B,N,H,d] storage, NaN codes behind the last key (transposed v: behind every row of keys), an output whose padding must stay untouched."""
    B, H, nq, nk, d, pad = 2, 3, 90, 1008, 96, 80
    q, k, v = _inputs(5, B, H, H, nq, nk, d, E4)

    def spread_out(t, rows_first):
        t = t.permute(0, 2, 1, 3) if rows_first else t
        shape = list(t.shape)
        shape[1 if rows_first else 3] += pad
        buf = torch.full(shape, 0x7F, dtype=torch.uint8, device=DEV)
        at = buf[:, :t.shape[1]] if rows_first else buf[..., :t.shape[3]]
        at.copy_(t.view(torch.uint8))
        return at.permute(0, 2, 1, 3).view(E4) if rows_first else at.view(E4)

    vv = v.transpose(2, 3).contiguous() if vt else v
    obuf = torch.full((B, nq + pad, H, d), 777.0, dtype=torch.float16, device=DEV)
    o = obuf[:, :nq].permute(0, 2, 1, 3)
    wide = spread_out(q, True), spread_out(k, True), spread_out(vv, not vt)  # (kept: the parameters hold pointers only)
    p = fa.make_params(*wide, o, True, 0.1, vt, causal_bottom_right=True)
    assert fa.lib().fa8_fwd_apart(ctypes.byref(p)) == 1
    assert fa.lib().fa8_fwd_any_order(ctypes.byref(p), None, 0, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    assert torch.equal(o.contiguous(), fa.flash_attention_v2_cutlass(q, k, vv, True, 0.1, v_transposed=vt, causal_bottom_right=True)[0])
    assert (obuf[:, nq:] == 777.0).all()


PAIRS = [
    # B, H, Hk, Nq, Nk, d, (rows per workgroup, wavefronts per tile): shifts of half a block, so that the second tile of a workgroup sees a block more
    (1, 30, 30, 1504, 1536, 32, (64, 2)),
    (1, 20, 20, 2080, 2112, 64, (64, 2)),
    (1, 28, 28, 1088, 1120, 96, (64, 2)),
    (1, 20, 20, 1600, 1632, 128, (64, 2)),
    (1, 30, 30, 320, 1376, 96, (64, 4)),
    (1, 30, 30, 320, 1376, 128, (64, 4)),
    (1, 32, 8, 504, 2048, 128, (64, 4)),  # group of 4, tiles of 8 queries: every fourth workgroup
]


@pytest.mark.parametrize("shape", PAIRS, ids=lambda s: "B{}H{}k{}Nq{}Nk{}d{}".format(*s[:6]))
@pytest.mark.parametrize("dt,code", [(E4, 0x7F), (E5, 0x7F), (E5, 0x7C)], ids=["e4m3-nan", "e5m2-nan", "e5m2-inf"])
@pytest.mark.parametrize("vt", [False, True], ids=["rows", "vt"])
def test_infinity_and_nan_in_v_stay_out_of_a_tile_that_ends_before_their_block(shape, dt, code, vt):
    """Two tiles a workgroup, mask aligned to the last key: a block that only the second tile sees holds an infinity or a NaN, its weights in the first
    are zero.  Rows that fa8_fwd gives finite are finite here too.  Another workgroup in every k/v head, so that the block falls to every wavefront."""
    B, H, Hk, Nq, Nk, d, cut = shape
    q, k, v = _inputs(7, B, H, Hk, Nq, Nk, d, dt)
    group, tile = H // Hk, 32 // (H // Hk)
    pairs = [p for p in range(Nq // (2 * tile)) if (2 * tile * p + tile + Nk - Nq) % 64 == 0]
    for head in range(Hk):
        first_key = 2 * tile * pairs[-1 - head % len(pairs)] + tile + Nk - Nq  # the first that the pair's first tile does not see
        v.view(torch.uint8)[0, head, first_key + (head % 3) * (tile // 2 - 1), 5 * head % d] = code
    fine_v = torch.where(torch.isfinite(v.float()), v.float(), torch.zeros(()).to(DEV))
    if vt:
        v = v.transpose(2, 3).contiguous()
    kw = dict(v_transposed=vt, return_lse=True, causal_bottom_right=True)
    got, lse = fa.flash_attention_v2_cutlass(q, k, v, True, d ** -0.5, **kw)
    want, want_lse = torch.empty_like(got), torch.empty_like(lse)
    p = fa.make_params(q, k, v, want, True, d ** -0.5, vt, want_lse, True)
    assert fa.lib().fa8_fwd_apart(ctypes.byref(p)) == 1 and fa.plan(p, fa.FA8_PLAN_ANY_ORDER) == cut + (1,)
    assert fa.lib().fa8_fwd(ctypes.byref(p), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    fine = torch.isfinite(want)
    assert 0 < (~fine).sum() < fine.numel() // 2
    assert torch.equal(torch.isfinite(got), fine) and torch.equal(torch.isnan(got), torch.isnan(want))
    assert_same_up_to_sum_order(got[fine], want[fine], fine_v, Nk)
    assert (lse - want_lse).abs().max() <= 5e-6 * max(1.0, want_lse.abs().max().item())


@pytest.mark.parametrize("shape,causal,br,vt,dt,rows", [
    ((1, 2, 2, 100, 705, 64), False, False, False, E4, None),
    ((1, 4, 2, 70, 784, 64), True, True, True, E5, None),
    ((2, 6, 2, 11, 900, 32), True, True, False, E4, None),
    ((1, 8, 4, 40, 1100, 96), True, True, False, E4, None),
    ((1, 3, 3, 200, 1232, 128), False, False, True, E4, None),
    ((1, 32, 32, 500, 760, 96), False, False, False, E4, 48),   # two tiles, four wavefronts
    ((1, 30, 30, 270, 1330, 128), True, True, False, E4, 48),
    ((1, 24, 24, 1300, 1300, 64), False, False, False, E4, 48),  # two tiles, two wavefronts
    ((1, 28, 28, 1088, 1120, 96), True, True, True, E5, 48),
    ((1, 20, 20, 1600, 1632, 128), True, True, False, E4, 48),
], ids=lambda x: "B{}H{}k{}Nq{}Nk{}d{}".format(*x) if isinstance(x, tuple) else "")
def test_sums_apart_against_the_oracle(shape, causal, br, vt, dt, rows):
    """The gate of every GPU parity test (max-abs 2e-2 a row, mean-abs 2e-3 against the oracle in the device's arithmetic), through the binding."""
    q, k, v = _inputs(shape[3] + shape[4], *shape, dt)
    vv = v.transpose(2, 3).contiguous() if vt else v
    scale = shape[5] ** -0.5
    o, lse = fa.load_extension().flash_attention_v2_cutlass(q, k, vv, causal, scale, v_transposed=vt, return_lse=True, causal_bottom_right=br)
    assert fa.lib().fa8_fwd_apart(ctypes.byref(fa.make_params(q, k, vv, o, causal, scale, vt, lse, br))) == 1
    at = None if rows is None else sample_rows(shape[3], rows)
    got, got_lse = o.float().cpu().numpy(), lse.cpu().numpy()
    _, want_lse = assert_parity(got if at is None else got[:, :, at], *(t.view(torch.uint8).cpu().numpy() for t in (q, k, v)), scale, causal=causal, rows=at,
                                kv_block=fa.query(fa.FA8_QUERY_KV_BLOCK), in_dtype=fo.E5M2 if dt == E5 else fo.E4M3, causal_bottom_right=br, label=f"apart {shape}")
    assert abs((got_lse if at is None else got_lse[:, :, at]) - want_lse).max() <= 5e-6 * max(1.0, abs(want_lse).max())
