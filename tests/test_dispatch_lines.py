"""CPU tests of where the planner's lines between kernels lie: shapes on both sides of each, measured on a
256-CU device (without a GPU the planner assumes one), as the plan that was the faster there."""
import pytest

from nebula_amd import hq

I4, T2, F16, BF16 = hq.FORMAT_INT4, hq.FORMAT_TERNARY2, hq.DTYPE_F16, hq.DTYPE_BF16


def plan(fmt, dt, M, K, N, **kw):
    import torch

    if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are those of a 256-CU device")
    return hq.describe(fmt, dt, M, K, N, **kw)


# Shared row tiles: slabs of four tiles that leave CUs idle lose over a long K, by rows.
@pytest.mark.parametrize("fmt,M,slabs,kblocks,rows", [
    (T2, 56, 130, 32, True), (T2, 56, 130, 48, False), (T2, 80, 130, 48, True), (T2, 80, 130, 96, False),
    (I4, 64, 160, 152, False), (I4, 56, 136, 151, False), (I4, 80, 86, 96, True), (I4, 80, 86, 128, False), (T2, 33, 86, 48, True),
    (T2, 33, 86, 96, False), (T2, 20, 86, 32, True), (T2, 20, 86, 64, False),
    (I4, 80, 172, 176, True), (T2, 56, 184, 128, True), (T2, 33, 172, 88, True), (T2, 33, 172, 112, False),  # past one lockstep workgroup per CU
    (T2, 20, 256, 32, True), (T2, 20, 256, 48, False), (T2, 33, 256, 64, True), (T2, 33, 256, 96, False),
    (T2, 56, 256, 96, True), (I4, 80, 256, 112, True), (I4, 80, 240, 176, True), (T2, 80, 240, 192, False), (T2, 33, 86, 64, True),
    (I4, 80, 32, 216, True), (T2, 56, 16, 216, True),                              # few slabs in eight pieces
])
def test_row_tiles_by_piece_length(fmt, M, slabs, kblocks, rows):
    assert plan(fmt, F16, M, 128 * kblocks, 64 * slabs).startswith("hq_rows_kernel<" if rows else "hq_decode_ls_kernel<")


def test_row_tiles_by_type():
    # Int4 with bf16, whose lockstep kernel carries a correction chain, keeps the row tiles longer; what a call
    # asks for is the same for both types.
    for M, kblocks, slabs in ((40, 88, 240), (56, 112, 240), (40, 76, 86)):
        f, b = (plan(I4, dt, M, 128 * kblocks, 64 * slabs) for dt in (F16, BF16))
        assert f.startswith("hq_decode_ls_kernel<") and b.startswith("hq_rows_kernel<"), (f, b)
        assert f.split(" ws=")[1] == b.split(" ws=")[1]


# Ternary prefill in groups of 64 past one 64 x 128 tile per CU: the 64-row tiles stay where their rounds of
# one tile per CU are cheaper.
@pytest.mark.parametrize("dt,group,M,kblocks,N,tile", [
    (BF16, 64, 643, 15, 23680, "64-row tiles=1023 whole"), (BF16, 64, 736, 17, 15360, "64-row tiles=720 whole"),
    (F16, 64, 736, 17, 15360, "128-row tiles=360"), (BF16, 64, 891, 46, 15360, "128-row tiles=420"),
])
def test_ternary_tiles_past_one_per_cu(dt, group, M, kblocks, N, tile):
    d = plan(T2, dt, M, 128 * kblocks, N, group=group)
    assert tile in d, d


# General int4 decode (group 32 with a bias): slabs that leave CUs idle, or need a second round, against
# the lockstep kernel's.
@pytest.mark.parametrize("M,kblocks,N,resident", [
    (16, 8, 24576, True), (16, 24, 24576, False), (9, 40, 24576, False), (16, 24, 23552, True), (4, 16, 24576, True),
    (4, 112, 10240, False), (2, 152, 10240, False), (4, 64, 10240, True), (1, 112, 9216, True),
    (4, 112, 4400, False), (1, 152, 4400, False), (4, 88, 4400, True), (6, 152, 4400, True),
    (4, 152, 5120, False), (4, 112, 5120, True), (4, 112, 2560, True),
])
def test_general_resident_slabs(M, kblocks, N, resident):
    d = plan(I4, BF16, M, 128 * kblocks, N, group=32, with_bias=True)
    assert d.startswith("hq_decode_xr_kernel<" if resident else "hq_decode_ls_kernel<"), d
    if (M, kblocks, N) == (16, 8, 24576):  # two workgroups of four wavefronts per CU
        assert "x 4 wavefronts" in d


def test_lockstep_keeps_fp32_scales_where_the_row_tiles_would_have_them():
    # Int4, fp16, 65 to 80 rows: a piece too long for the row tiles must not round its weights times their scales.
    assert " fp32 scales" in plan(I4, F16, 80, 19456, 8320)
    for fmt, dt, M, K, N in ((I4, F16, 80, 5120, 34816), (I4, BF16, 80, 19456, 8320), (I4, F16, 64, 19456, 8320)):
        assert plan(fmt, dt, M, K, N).startswith("hq_decode_ls_kernel<") and " fp32 scales" not in plan(fmt, dt, M, K, N)
