"""GPU tests of the prefill kernel's 128-column tiles whose k-blocks are split between groups of
wavefronts of one workgroup (64 x 128 tiles in two or four groups, 128 x 128 in two), and the
general kernels' 128-row tiles, forced on ragged shapes and as the planner picks them."""
import pytest

import oracle as O
from gpu_util import DeviceProblem
from nebula_amd import hq
from test_gpu_general import Dev
from test_gpu_general import check as check_general
from test_gpu_parity import check

pytestmark = pytest.mark.gpu

FMTS = [(O.INT4, O.F16), (O.INT4, O.BF16), (O.TERNARY2, O.F16), (O.TERNARY2, O.BF16)]


# RT * 100 + KS * 10 + TW. K: k-blocks that do not divide by the groups, and one to a group; N: one
# column, a tile boundary, a ragged last block; M: around the tile heights.
@pytest.mark.parametrize("tile", [442, 422, 822])
@pytest.mark.parametrize("fmt,xdt", FMTS)
@pytest.mark.parametrize("M,K,N", [(65, 512, 1), (64, 640, 128), (127, 896, 250), (129, 1408, 257)])
def test_forced_tiles(cuda, monkeypatch, tile, fmt, xdt, M, K, N):
    from test_gpu_parity import torch_equal

    monkeypatch.setenv("HQ_PREFILL_TILE", str(tile))
    monkeypatch.setenv("HQ_DECODE_MAX_M", "16")
    P = O.Problem(fmt, M, K, N, 128, xdt, seed=8900 + M)
    assert "k-split in workgroup" in hq.describe(fmt, xdt, M, K, N)
    D = DeviceProblem(P)
    y = D.run()
    assert torch_equal(y, D.run())  # the groups' sums meet in group order
    check(y, P.reference(), xdt, f"tile={tile} fmt={fmt} dt={xdt} M={M} K={K} N={N}", P)


@pytest.mark.parametrize("tile", [442, 422, 822, 814, 812])
@pytest.mark.parametrize("fmt,xdt,g,bias", [(O.INT4, O.F16, 32, "random"), (O.INT4, O.BF16, 64, "random"),
                                            (O.INT4, O.F16, 64, None), (O.INT4, O.BF16, 32, None),
                                            (O.TERNARY2, O.F16, 32, None), (O.TERNARY2, O.BF16, 64, None)])
@pytest.mark.parametrize("M,K,N", [(66, 512, 130), (129, 1408, 257)])
def test_forced_tiles_general(cuda, monkeypatch, tile, fmt, xdt, g, bias, M, K, N):
    monkeypatch.setenv("HQ_PREFILL_TILE", str(tile))
    monkeypatch.setenv("HQ_DECODE_MAX_M", "16")
    P = O.Problem(fmt, M, K, N, g, xdt, seed=8950 + M, bias=bias)
    check_general(Dev(P).run(), P, f"general tile={tile} fmt={fmt} dt={xdt} g={g} M={M}")


def test_fused_segments_and_strides(cuda, monkeypatch):
    # Blocks of several segments, an output row stride of its own, columns past N untouched.
    import torch

    monkeypatch.setenv("HQ_PREFILL_TILE", "442")
    M, K, Ns = 100, 1152, [130, 16, 300]
    probs = [O.Problem(O.INT4, M, K, n, 128, O.F16, seed=8990 + i) for i, n in enumerate(Ns)]
    for p in probs[1:]:
        p.X = probs[0].X
    devs = [DeviceProblem(p) for p in probs]
    wide = [torch.full((M, n + 7), 3.0, dtype=torch.float16, device="cuda") for n in Ns]
    hq.gemm_fused(O.INT4, devs[0].X, [(d.Wp, d.S, d.P.N) for d in devs], outs=[w[:, :n] for w, n in zip(wide, Ns)])
    for d, w, n in zip(devs, wide, Ns):
        check(w[:, :n], d.P.reference(), O.F16, f"fused N={n}", d.P)
        assert bool((w[:, n:] == 3.0).all())


@pytest.mark.parametrize("fmt,M,K,N,g,want", [
    (O.INT4, 128, 4096, 14336, 128, "64x128 tiles=224 whole=224 stream-K workgroups=0 four-way"),
    (O.INT4, 384, 1024, 4096, 128, "64x128 tiles=192 whole=192 stream-K workgroups=0 k-split"),
    (O.INT4, 256, 4096, 14336, 128, "128-row 128-column tiles=224 whole=224 stream-K workgroups=0 k-split"),
    (O.TERNARY2, 256, 4096, 14336, 128, "64x128 tiles=448"),
    (O.INT4, 192, 4096, 20480, 128, "64x128 tiles=480"),
    (O.INT4, 96, 4096, 1024, 128, "whole=0 stream-K"),          # 16 tiles: the K split over workgroups
    (O.TERNARY2, 256, 14336, 4096, 128, "whole=0 stream-K"),    # a long K
    (O.TERNARY2, 400, 6144, 5120, 256, "whole=0 stream-K"),
    (O.INT4, 1024, 4096, 14336, 32, "general> launch 0: 128-row tiles=448"),
    (O.INT4, 512, 4096, 14336, 32, "general> launch 0: 128-row 128-column tiles=448"),
])
def test_default_plans(cuda, fmt, M, K, N, g, want):
    import torch

    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the boundaries are those of a 256-CU device")
    for dt in (O.F16, O.BF16):
        assert want in hq.describe(fmt, dt, M, K, N, group=g)


# Whole 64 x 128 tiles against the K split over workgroups, by cost (the planner needs the device's occupancy for
# the split): shapes measured 5% and more apart, where K divides well, badly, and with ragged rows.
@pytest.mark.parametrize("fmt,dt,group,M,kblocks,N,whole", [
    (O.INT4, O.BF16, 128, 81, 112, 7168, False), (O.INT4, O.BF16, 128, 300, 216, 4096, False), (O.INT4, O.BF16, 128, 512, 70, 1408, True),
    (O.INT4, O.BF16, 128, 768, 160, 2176, True), (O.INT4, O.F16, 128, 81, 112, 7168, True), (O.INT4, O.F16, 128, 96, 64, 5120, True),
    (O.TERNARY2, O.F16, 128, 226, 80, 3072, False), (O.TERNARY2, O.F16, 128, 226, 76, 2560, True),
    (O.TERNARY2, O.BF16, 128, 81, 76, 5120, True), (O.TERNARY2, O.F16, 128, 300, 64, 2048, True),
    (O.TERNARY2, O.BF16, 128, 747, 128, 461, True), (O.TERNARY2, O.BF16, 64, 300, 27, 2048, True),
    (O.INT4, O.BF16, 32, 1024, 200, 1792, True),
])
def test_small_tiles_by_cost(cuda, fmt, dt, group, M, kblocks, N, whole):
    import torch

    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the boundaries are those of a 256-CU device")
    d = hq.describe(fmt, dt, M, 128 * kblocks, N, group=group, with_bias=group == 32)
    assert ("64x128 tiles=" if whole else "whole=0 stream-K") in d, d
    assert d.split(" ws=")[1] == hq.describe(fmt, O.F16 + O.BF16 - dt, M, 128 * kblocks, N, group=group, with_bias=group == 32).split(" ws=")[1]


# Three equal pieces along K (the planner needs the device's occupancy for them): ternary fp16, and both
# types in groups of 64, stay split; pieces that do not come out equal take the whole tiles.
@pytest.mark.parametrize("dt,group,M,kblocks,N,split", [
    (O.F16, 128, 300, 36, 7168, True), (O.BF16, 128, 300, 36, 7168, False), (O.F16, 128, 300, 35, 7168, False),
    (O.F16, 128, 300, 36, 8704, False), (O.F16, 64, 167, 36, 14336, True), (O.BF16, 64, 1762, 39, 1280, True),
    (O.BF16, 64, 167, 37, 14336, False), (O.BF16, 64, 300, 27, 7168, False),
])
def test_three_equal_pieces_stay_split(cuda, dt, group, M, kblocks, N, split):
    import torch

    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the boundaries are those of a 256-CU device")
    d = hq.describe(O.TERNARY2, dt, M, 128 * kblocks, N, group=group)
    assert ("whole=0 stream-K" if split else "64x128 tiles=") in d, d


# The plans of test_default_plans as they run, the new tiles at the sizes they serve: grids of 192 to 480 tiles over
# several row bands, four groups over 32 and more k-blocks, the general 128-row tiles over more than one
# round. Each row band's first and last row and a few between are compared.
@pytest.mark.parametrize("fmt,xdt,M,K,N,group,bias", [
    (O.INT4, O.F16, 128, 4096, 14336, 128, None), (O.INT4, O.BF16, 384, 1024, 4096, 128, None),
    (O.INT4, O.BF16, 256, 4096, 14336, 128, None), (O.TERNARY2, O.F16, 256, 4096, 14336, 128, None),
    (O.TERNARY2, O.BF16, 192, 6144, 20480, 256, None), (O.INT4, O.F16, 192, 4096, 20480, 128, None),
    (O.INT4, O.F16, 1024, 4096, 14336, 32, "random"), (O.INT4, O.BF16, 1024, 4096, 14336, 32, "random"),
    (O.INT4, O.F16, 512, 4096, 14336, 32, "random"), (O.INT4, O.BF16, 512, 4096, 14336, 64, "random"),
    (O.INT4, O.F16, 600, 1024, 28000, 32, "random"),
])
def test_default_plans_compute(cuda, fmt, xdt, M, K, N, group, bias):
    import numpy as np

    d = hq.describe(fmt, xdt, M, K, N, group=group, with_bias=bias is not None)
    assert "whole=0" not in d, d
    P = O.Problem(fmt, M, K, N, group, xdt, seed=8700 + M, bias=bias)
    rows = np.unique(np.concatenate([np.arange(0, M, 64), np.arange(63, M, 64), [M // 2 + 5, M - 1]]))
    y = Dev(P).run(bias=bias is not None)
    check_general(y, P, f"{d} M={M} K={K} N={N}", rows=rows)
