"""Full attention over keys that end inside a KV block: the dense loop with a masked last block.  The same arithmetic in the same order as
the rolling loop, so the results are compared bit for bit: every number of blocks up to two trips of its unrolled loop, ends on both sides
of the rows that the two passes of a tile copy take, both v layouts, guard bands behind the last key, infinities and NaN."""
import ctypes

import pytest
import torch

import cutlass_flash_atten_fp8_amd as fa

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
E4, E5 = torch.float8_e4m3fn, torch.float8_e5m2


def _guarded(t, rows):
    """The same values with NaN codes behind row `rows` - 1 of every head (a read past the last key would show)."""
    B, H, n, d = t.shape
    buf = torch.full((B, H, n + 70, d), 0x7F, dtype=torch.uint8, device=DEV)
    buf[:, :, :n] = t.view(torch.uint8)
    return buf.view(t.dtype)[:, :, :rows]


def _both(q, k, v, vt, out_dtype=torch.float16):
    res = []
    for schedule in (fa.FA8_SCHEDULE_ROLLING, fa.FA8_SCHEDULE_DENSE):
        o = torch.empty(q.shape, dtype=out_dtype, device=DEV)
        lse = torch.empty(q.shape[:3], device=DEV)
        p = fa.make_params(q, k, v, o, False, 0.125, vt, lse, False, schedule)
        assert fa.lib().fa8_fwd_schedule(ctypes.byref(p)) == schedule  # over keys that end inside a block: the masked form
        rc = fa.lib().fa8_fwd(ctypes.byref(p), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, fa.error_string(rc)
        res.append((o.float(), lse))
    torch.cuda.synchronize()
    return res


def _assert_same(res):
    for want, got in zip(*res):
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        assert torch.equal(got[~torch.isnan(got)], want[~torch.isnan(want)])


# head dim 64 takes the dense loop above three 128-row workgroups a compute unit (52 x 16 of them), head dim 128 always
@pytest.mark.parametrize("d,heads", [(128, 3), (64, 52 * 16)])
@pytest.mark.parametrize("keys", [1, 15, 16, 17, 32, 33, 48, 49, 63, 65, 127, 129, 160, 191, 193, 250, 257, 321, 391, 449, 511])
def test_every_number_of_blocks(d, heads, keys):
    g = torch.Generator(device=DEV).manual_seed(keys)
    q, k, v = ((3 * torch.randn(1, heads, n, d, device=DEV, generator=g)).to(E4) for n in (45, keys, keys))
    _assert_same(_both(q, _guarded(k, keys), _guarded(v, keys), False))


@pytest.mark.parametrize("d,heads", [(128, 3), (64, 52 * 16)])
@pytest.mark.parametrize("keys", [16, 48, 80, 112, 176, 208, 336])
def test_transposed_v(d, heads, keys):
    g = torch.Generator(device=DEV).manual_seed(keys)
    q, k, v = ((3 * torch.randn(1, heads, n, d, device=DEV, generator=g)).to(E5) for n in (45, keys, keys))
    vt = v.transpose(2, 3).contiguous()
    _assert_same(_both(q, _guarded(k, keys), vt, True, E5))


@pytest.mark.parametrize("keys,stride", [(65, 22486736), (79, 20950000), (100, 19004272)])
def test_rows_so_far_apart_that_a_second_copy_lies_past_31_bits(keys, stride):
    """The largest row strides that the library takes for so few keys: with 65 of them the second copy of the last block's V would start at
    2.16e9 bytes.  Between the rows lie NaN codes."""
    g = torch.Generator(device=DEV).manual_seed(keys)
    q, k, v = ((3 * torch.randn(1, 1, n, 128, device=DEV, generator=g)).to(E4) for n in (45, keys, keys))
    far = []
    for t in (k, v):
        buf = torch.full(((keys - 1) * stride + 128,), 0x7F, dtype=torch.uint8, device=DEV)
        rows = buf.as_strided((1, 1, keys, 128), (keys * stride, keys * stride, stride, 1))
        rows.copy_(t.view(torch.uint8))
        far.append(rows.view(E4))
    res = _both(q, *far, False)
    _assert_same(res)
    for want, got in zip(_both(q, k, v, False)[1], res[1]):
        assert torch.isfinite(got).all() and torch.equal(got, want)


@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("row", [3, 68, 199])
@pytest.mark.parametrize("code", [0x7C, 0x7F], ids=["inf", "nan"])  # of e5m2
def test_infinity_and_nan(where, row, code):
    g = torch.Generator(device=DEV).manual_seed(row)
    q, k, v = (torch.randn(1, 4, n, 128, device=DEV, generator=g).to(E5) for n in (200, 200, 200))
    {"q": q, "k": k, "v": v}[where].view(torch.uint8)[0, 1, row, 17] = code
    _assert_same(_both(q, k, v, False))


def test_first_block_of_keys_that_no_query_sees():
    """Keys of -inf in front (every logit -inf): the later keys alone decide."""
    g = torch.Generator(device=DEV).manual_seed(1)
    q, k, v = (torch.randn(1, 2, n, 128, device=DEV, generator=g).to(E5) for n in (40, 150, 150))
    q.view(torch.uint8)[:, :, :, 5] = 0x3C   # 1.0
    k.view(torch.uint8)[:, :, :64, 5] = 0xFC  # -inf
    res = _both(q, k, v, False)
    assert torch.isfinite(res[1][0]).all()
    _assert_same(res)
