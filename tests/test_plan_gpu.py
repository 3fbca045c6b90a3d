"""How a launch is cut (fa8_fwd_plan): rows of a workgroup, wavefronts per 32 rows, parts of the keys.  Launches that sharing a row tile makes
slower stay with one wavefront per tile.  Times: us on a MI355X, unshared / shared as the library once chose."""
import pytest
import torch

import cutlass_flash_atten_fp8_amd as fa

pytestmark = pytest.mark.gpu
UNSHARED = (128, 1, 1)


def params_of(B, H, Hk, Nq, Nk, d, causal=False, bottom_right=False, vt=False):
    """Nothing is launched: the parameters of tiny tensors with other sizes and contiguous strides."""
    t = torch.zeros((1, 1, 1, 256), dtype=torch.float8_e4m3fn, device="cuda:0")
    p = fa.make_params(t, t, t, torch.zeros((1, 1, 1, 256), dtype=torch.float16, device="cuda:0"), causal, d ** -0.5, vt, None, bottom_right)
    p.batch, p.heads, p.heads_k, p.seqlen_q, p.seqlen_k, p.head_dim = B, H, Hk, Nq, Nk, d
    for name, heads, rows, cols in (("q", H, Nq, d), ("k", Hk, Nk, d), ("v", Hk) + ((d, Nk) if vt else (Nk, d)), ("o", H, Nq, d)):
        setattr(p, name + "_row_stride", cols)
        setattr(p, name + "_head_stride", rows * cols)
        setattr(p, name + "_batch_stride", heads * rows * cols)
    return p


def plan_of(*shape, with_workspace=True):
    return fa.plan(params_of(*shape), with_workspace)


@pytest.mark.parametrize("shape", [
    (32, 32, 32, 288, 1024, 256),       # 249 / 559
    (64, 64, 64, 257, 1024, 64),        # 349 / 577
    (64, 64, 64, 288, 288, 128),        # 241 / 405
    (64, 64, 64, 96, 96, 96),           # 42 / 65
    (32, 32, 32, 192, 192, 96),         # 28.8 / 38.7
    (16, 70, 35, 192, 192, 128),        # 37.4 / 51.4
    (64, 64, 64, 33, 33, 96),           # 23.8 / 35.7: a single block
    (8, 32, 32, 64, 64, 64),            # 3.8 / 5.1
    (1, 1, 1, 1, 1, 128),               # 3.8 / 4.4
    (8, 12, 12, 157, 157, 128, True),   # 7.0 / 11.5: three blocks, 240 pairs
    (4, 17, 17, 224, 224, 96, True),    # 7.9 / 10.5
], ids=lambda s: "B{}H{}k{}Nq{}Nk{}d{}".format(*s[:6]))
def test_sharing_does_not_take_launches_that_it_slows_down(shape):
    if shape[4] <= 64 or shape[0] > 8:
        assert plan_of(*shape) == UNSHARED
    else:  # two wavefronts a tile: 7.1 and 6.4 us
        assert plan_of(*shape)[1] <= 2


@pytest.mark.parametrize("shape", [
    (1, 64, 64, 895, 1841, 128, True, True),   # 36.9 / 43.0: 3.5 pairs a compute unit, work of 2.7
    (1, 64, 64, 884, 1271, 128, True, True),   # 27.8 / 31.9
    (1, 32, 32, 1757, 3649, 96, True, True),   # 60.7 / 67.7
], ids=lambda s: "B{}H{}k{}Nq{}Nk{}d{}".format(*s[:6]))
def test_chunks_whose_tiles_are_long_throughout_are_not_shared(shape):
    assert plan_of(*shape) == UNSHARED


@pytest.mark.parametrize("shape", [
    (1, 1, 1, 32, 1121, 128, True, True),    # 10.0 shared, 19.3 split
    (1, 4, 1, 15, 1244, 64, True, True),     # 9.1, 16.7
    (1, 2, 1, 1051, 1051, 192, True),        # 15, 26.7
    (1, 2, 2, 1792, 1792, 160),              # 20.1, 35.5
    (1, 6, 2, 12, 1245, 128, True, True),    # 10.3, 18
    (4, 1, 1, 832, 1665, 160),               # 20.1, 34.1
    (4, 4, 4, 1, 974, 128, True, True),      # 8.8, 9.9: 16 blocks
    (1, 12, 6, 2, 999, 128, True, True),     # 8.6, 9.6
], ids=lambda s: "B{}H{}k{}Nq{}Nk{}d{}".format(*s[:6]))
def test_few_keys_are_not_split(shape):
    assert plan_of(*shape)[1:] == (4, 1)


def test_keys_are_not_split_where_their_bytes_bound_both():
    """16 sequences of 8191 keys, K and V from HBM: 53 us shared, at the rate of a plain copy, 69 split."""
    assert plan_of(16, 32, 8, 1, 8191, 128, True, True)[1:] == (4, 1)


@pytest.mark.parametrize("shape", [(1, 32, 8, 1, 32768, 128, True, True), (4, 32, 8, 1, 4096, 128, True, True), (1, 8, 8, 1, 4096, 64, True, True),
                                   (1, 2, 2, 16, 4096, 224),
                                   # K and V bound by few bytes under way with one LDS stage: 105 us shared, 82 split; 129, 101; 156, 132; 173, 151
                                   (64, 4, 2, 1, 7695, 192, True, True), (2, 64, 64, 2, 9601, 192, True, True),
                                   (16, 12, 6, 2, 11470, 256, True, True), (8, 12, 12, 2, 42156, 64, True, True)], ids=lambda s: "B{}H{}k{}Nq{}Nk{}d{}".format(*s[:6]))
def test_many_keys_are_split(shape):
    assert plan_of(*shape)[2] > 1 and plan_of(*shape, with_workspace=False)[2] == 1


def test_head_counts_beyond_32_bit_products():
    """65535 sequences of 1024 heads on one k/v head: 40 * batch * heads does not fit 32 bits; one query each leaves 127 of 128 rows idle."""
    assert plan_of(65535, 1024, 1, 1, 1, 128) == (64, 2, 1)


@pytest.mark.parametrize("shape,name", [
    ((1, 20, 20, 1600, 1632, 128, True, True), "shared rows (2 wavefronts, sums apart)"),  # where fa8_fwd_ws runs a main loop
    ((1, 16, 16, 1024, 1024, 64, True), "shared rows (4 wavefronts, sums apart)"),
    ((1, 16, 16, 128, 128, 64), "shared rows (4 wavefronts)"),
    ((1, 32, 8, 1, 32768, 128, True, True), "split keys (32 parts)"),
    ((2, 32, 32, 4096, 4096, 128), "dense"),
], ids=lambda s: "B{}H{}k{}Nq{}Nk{}d{}".format(*s[:6]) if isinstance(s, tuple) else "")
def test_the_benchmark_names_what_a_call_through_the_binding_runs(shape, name):
    import bench
    assert bench.loop_name(fa, params_of(*shape)) == name
