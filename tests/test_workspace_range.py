"""CPU tests of the workspace a call asks for where kernels that write no partial sums take some of
the rows between 1 and 80, or some prefill grids: a buffer sized at the largest batch keeps serving
the smaller ones, as it did with the kernels that cut these shapes along K."""
import ctypes

import pytest

from nebula_amd import hq

ROWS = [17, 32, 33, 48, 49, 64, 65, 80]


def need(fmt, M, K, Ns, group=128, bias=0):
    return hq.workspace_bytes_fused(fmt, M, K, Ns, group, bool(bias))


# Slabs that fill half to two thirds of the CUs, a long K, few slabs, one per CU, segments, ragged widths.
SHAPES = [(27648, [5120]), (28672, [8192]), (9984, [10496]), (14208, [3528, 588, 588]), (5888, [13829]), (4096, [4096]),
          (17408, [5120]), (20992, [8704]), (5120, [9000]), (5120, [14336]), (1408, [315]), (5120, [34816])]


@pytest.mark.parametrize("fmt", [hq.FORMAT_INT4, hq.FORMAT_TERNARY2])
@pytest.mark.parametrize("K,Ns", SHAPES)
def test_need_does_not_fall_with_the_rows_up_to_80(fmt, K, Ns):
    sizes = [need(fmt, M, K, Ns) for M in ROWS]
    assert sizes == sorted(sizes), list(zip(ROWS, sizes))
    assert max(need(fmt, M, K, Ns) for M in (1, 2, 4, 8, 9, 16)) <= sizes[-1]


@pytest.mark.parametrize("K,Ns", SHAPES)
def test_need_of_general_int4_calls_does_not_fall_with_the_rows(K, Ns):
    sizes = [need(hq.FORMAT_INT4, M, K, Ns, 32, bias=1) for M in [1, 2, 4, 8, 9, 16] + ROWS]
    assert sizes == sorted(sizes)


@pytest.mark.parametrize("fmt,K,Ns,group,bias", [(hq.FORMAT_TERNARY2, 3328, [512], 128, 0), (hq.FORMAT_INT4, 4096, [4096], 128, 0),
                                                 (hq.FORMAT_INT4, 10496, [92, 16, 16], 128, 0), (hq.FORMAT_INT4, 1408, [315], 32, 1),
                                                 (hq.FORMAT_TERNARY2, 7936, [7362], 64, 0), (hq.FORMAT_INT4, 4096, [14336], 32, 1)])
def test_prefill_asks_for_what_the_256_column_plan_does(monkeypatch, fmt, K, Ns, group, bias):
    Ms = (81, 128, 192, 256, 333, 512, 1024, 2048)
    asked = [need(fmt, M, K, Ns, group, bias) for M in Ms]
    monkeypatch.setenv("HQ_PREFILL_TW", "1")  # the plan over 256-column tiles stays
    assert asked == [need(fmt, M, K, Ns, group, bias) for M in Ms]
    assert any(asked)


def test_a_plan_that_writes_nothing_takes_any_workspace():
    # Ternary 11264 x 11008 at 80 rows runs whole slabs: it asks for what 20 rows need, but does not refuse
    # a smaller buffer. At 20 rows, pieces: one byte less is refused (before any launch).
    L = hq.lib()
    K, N = 11264, 11008
    big, small = need(hq.FORMAT_TERNARY2, 80, K, [N]), need(hq.FORMAT_TERNARY2, 20, K, [N])
    assert big >= small > 0
    assert "hq_rows_kernel" in hq.describe(hq.FORMAT_TERNARY2, hq.DTYPE_F16, 80, K, N)
    segs = (hq.Segment * 1)(hq.Segment(0x2000, 0x3000, None, 0x4000, N, N))
    args = (0x1000, hq.DTYPE_F16, K, hq.FORMAT_TERNARY2, segs, 1, 20, K, 128)
    assert L.hq_gemm_fused(*args, ctypes.c_void_p(0x10000), small - 1, None) == hq.HQ_ERR_WORKSPACE
    assert L.hq_gemm_fused(*args, ctypes.c_void_p(0x10010), big, None) == hq.HQ_ERR_ALIGNMENT
