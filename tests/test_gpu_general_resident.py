"""GPU tests of the X-resident decode kernel's general int4 form (groups that are multiples of 32,
an optional bias): every slab width it has, wavefronts without k-blocks, pieces along K, ragged
columns, segments with and without a bias, and the plans the library picks."""
import pytest

import oracle as O
from gpu_util import to_host_f32
from nebula_amd import hq
from test_gpu_general import Dev, check, env

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,WK,S", [(1, 8, 1), (2, 8, 1), (4, 8, 1), (4, 4, 1), (4, 1, 1), (2, 5, 3), (4, 8, 2)])
@pytest.mark.parametrize("xdt,g,bias", [(O.F16, 32, "random"), (O.BF16, 32, "random"), (O.F16, 96, None),
                                        (O.BF16, 128, "random")])
def test_forced_slabs(cuda, T, WK, S, xdt, g, bias):
    for M, K, N in ((1, 384, 530), (7, 768, 515), (16, 1152, 4112)):
        P = O.Problem(O.INT4, M, K, N, g, xdt, seed=9300 + M, bias=bias)
        with env(HQ_XR_T=T, HQ_XR_WK=WK, HQ_XR_S=S):
            desc = hq.describe(O.INT4, xdt, M, K, N, group=g, with_bias=bias is not None)
            assert desc.startswith("hq_decode_xr_kernel<") and ",general>" in desc and f"x {S} pieces" in desc, desc
            D = Dev(P)
            y = D.run()
            assert bool((y == D.run()).all())  # one order of sums
        check(y, P, f"general resident T={T} WK={WK} S={S} dt={xdt} g={g} M={M}")


# Few tiles, a CU each, 4-tile slabs one to a CU and past one round, pieces of a long K.
@pytest.mark.parametrize("M,K,N", [(3, 4096, 512), (8, 1024, 4096), (4, 1024, 14336), (16, 512, 14336), (5, 512, 27648),
                                   (4, 27648, 1024), (8, 14336, 4096)])
def test_default_plans(cuda, M, K, N):
    P = O.Problem(O.INT4, M, K, N, 32, O.BF16, seed=9350 + M, bias="random")
    assert hq.describe(O.INT4, O.BF16, M, K, N, group=32, with_bias=True).startswith("hq_decode_xr_kernel<")
    check(Dev(P).run(), P, f"general resident M={M} K={K} N={N}")


# Nine to 16 rows over at most one tile per CU: one-tile slabs, ragged columns, an odd k-block count.
@pytest.mark.parametrize("xdt", [O.F16, O.BF16])
@pytest.mark.parametrize("M,K,N,g,bias", [(9, 1024, 4096, 32, "random"), (16, 2816, 1530, 64, None), (12, 4096, 4090, 32, "random"),
                                          (16, 5120, 2048, 32, "random"), (13, 14336, 512, 32, "random")])
def test_default_plans_of_nine_to_sixteen_rows(cuda, xdt, M, K, N, g, bias):
    P = O.Problem(O.INT4, M, K, N, g, xdt, seed=9360 + M, bias=bias)
    assert hq.describe(O.INT4, xdt, M, K, N, group=g, with_bias=bias is not None).startswith("hq_decode_xr_kernel<")
    D = Dev(P)
    y = D.run()
    assert bool((y == D.run()).all())
    check(y, P, f"general resident M={M} K={K} N={N} dt={xdt}")


def test_segments_with_and_without_bias(cuda):
    import torch

    M, K, Ns = 6, 1024, [530, 64, 700]
    probs = [O.Problem(O.INT4, M, K, n, 64, O.F16, seed=9380 + i, bias="random" if i != 1 else None) for i, n in enumerate(Ns)]
    for p in probs[1:]:
        p.X = probs[0].X
    devs = [Dev(p) for p in probs]
    segs = [(d.Wp, d.S, d.P.N, d.B if d.P.bias is not None else None) for d in devs]
    outs = hq.gemm_fused(O.INT4, devs[0].X, segs, 64)
    alone = [d.run(bias=d.P.bias is not None) for d in devs]
    for d, y, z in zip(devs, outs, alone):
        check(y, d.P, f"segment N={d.P.N}")
        assert O.normwise_error(to_host_f32(y), to_host_f32(z)) <= 1e-3
    assert torch.isfinite(outs[1]).all()
