"""GPU tests of the shared-row-tile kernel (17 <= M <= 80): every row-tile count, format and type, pieces
along K, k-groups without k-blocks, ragged columns, segments, strides, and the plans the library picks."""
import numpy as np
import pytest

import oracle as O
from gpu_util import DeviceProblem, to_dev_u16, to_host_f32
from nebula_amd import hq
from test_gpu_parity import check, torch_equal

pytestmark = pytest.mark.gpu

FMTS = [(O.INT4, O.F16), (O.INT4, O.BF16), (O.TERNARY2, O.F16), (O.TERNARY2, O.BF16)]


# K: one k-block (three idle k-groups), a remainder, a deeper ring; N: one column, tile and slab edges.
@pytest.mark.parametrize("fmt,xdt", FMTS)
@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64, 65, 80])
def test_row_tiles(cuda, monkeypatch, fmt, xdt, M):
    for K, N, S in ((128, 1, 1), (640, 129, 1), (1408, 200, 3), (2304, 66, 5), (384, 64, 3)):
        monkeypatch.setenv("HQ_ROWS", str(S))
        P = O.Problem(fmt, M, K, N, 128, xdt, seed=9500 + M)
        assert hq.describe(fmt, xdt, M, K, N).startswith("hq_rows_kernel<")
        D = DeviceProblem(P)
        y = D.run()
        assert torch_equal(y, D.run())  # one order of sums
        check(y, P.reference(), xdt, f"rows fmt={fmt} dt={xdt} M={M} K={K} N={N} S={S}", P)


@pytest.mark.parametrize("fmt,M,K,N,group,rows", [
    (O.TERNARY2, 80, 6144, 5120, 256, True), (O.TERNARY2, 20, 4096, 4096, 256, True), (O.INT4, 37, 4096, 11008, 128, True),
    (O.INT4, 80, 8192, 2048, 512, True),
    (O.INT4, 32, 4096, 11008, 128, False),      # int4 up to 32 rows
    (O.TERNARY2, 20, 5120, 9000, 128, False),   # 141 slabs at few rows
    (O.TERNARY2, 20, 17408, 5120, 256, False),  # a long K at few rows
    (O.TERNARY2, 80, 5120, 34816, 256, False),  # more slabs than CUs
])
def test_default_plans(cuda, fmt, M, K, N, group, rows):
    import torch

    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the boundaries are those of a 256-CU device")
    for xdt in (O.F16, O.BF16):
        assert hq.describe(fmt, xdt, M, K, N, group=group).startswith("hq_rows_kernel<" if rows else "hq_decode_ls_kernel<")
    if rows:
        P = O.Problem(fmt, M, K, N, group, O.BF16, seed=9600 + M)
        check(DeviceProblem(P).run(), P.reference(threads=16), O.BF16, f"rows default M={M} K={K} N={N}", P)


# Pieces one k-block too long for the row tiles: the lockstep kernel, whose int4 fp16 form at five row tiles keeps
# the scales in fp32 there. Its error in the 2-norm is the rounding of the outputs to fp16, uniform over an ulp: 2^-10 /
# sqrt(12) of the binade's foot, 1.9e-4 to 2.1e-4 of the values. Rounding the products of weight and scale adds as
# much again, independently, 2.8e-4 in all: the line is halfway.
@pytest.mark.parametrize("M,Ns", [(65, [8250]), (80, [8250]), (80, [5000, 1000, 2250])])
def test_long_pieces_keep_fp32_scales(cuda, M, Ns):
    import torch

    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the boundaries are those of a 256-CU device")
    K = 128 * 65
    if len(Ns) == 1:
        assert " fp32 scales" in hq.describe(O.INT4, O.F16, M, K, Ns[0])
    probs = [O.Problem(O.INT4, M, K, n, 128, O.F16, seed=9640 + i) for i, n in enumerate(Ns)]
    for p in probs:
        p.X = probs[0].X
    devs = [DeviceProblem(p) for p in probs]
    segs = [(d.Wp, d.S, d.P.N) for d in devs]
    outs = hq.gemm_fused(O.INT4, devs[0].X, segs)
    for p, y, z in zip(probs, outs, hq.gemm_fused(O.INT4, devs[0].X, segs)):
        assert torch_equal(y, z)  # one order of sums
        ref = p.reference(threads=16)
        check(y, ref, O.F16, f"fp32 scales M={M} N={p.N}", p)
        e = to_host_f32(y).astype(np.float64) - ref
        assert np.linalg.norm(e) <= 2.4e-4 * np.linalg.norm(ref.astype(np.float64))


def test_non_finite_scales_strides_and_counters(cuda, monkeypatch):
    # Ternary groups without a finite scale drop out; X and Y have row strides of their own; a caller
    # workspace is left with zero counters and serves two calls.
    import torch

    monkeypatch.setenv("HQ_ROWS", "3")
    M, K, Ns = 70, 1152, [130, 16, 300]
    probs = [O.Problem(O.TERNARY2, M, K, n, 128, O.F16, seed=9650 + i) for i, n in enumerate(Ns)]
    for p in probs:
        p.X = probs[0].X
        p.scales = p.scales.copy()
        p.scales[1, ::3], p.scales[2, 1::5] = np.uint16(0x7C00), np.uint16(0x7E01)
    devs = [DeviceProblem(p) for p in probs]
    Xw = torch.zeros((M, K + 64), dtype=torch.float16, device="cuda")
    Xw[:, :K] = to_dev_u16(probs[0].X, O.F16)
    ws = torch.zeros(hq.workspace_bytes_fused(O.TERNARY2, M, K, Ns), dtype=torch.uint8, device="cuda")
    assert ws.numel() > 65536
    for _ in range(2):
        wide = [torch.full((M, n + 5), 3.0, dtype=torch.float16, device="cuda") for n in Ns]
        hq.gemm_fused(O.TERNARY2, Xw[:, :K], [(d.Wp, d.S, d.P.N) for d in devs], outs=[w[:, :n] for w, n in zip(wide, Ns)],
                      workspace=ws)
        for d, w, n in zip(devs, wide, Ns):
            check(w[:, :n], d.P.reference(), O.F16, f"rows fused N={n}", d.P)
            assert bool((w[:, n:] == 3.0).all())
    assert int(ws[:65536].view(torch.int32).abs().sum().item()) == 0
