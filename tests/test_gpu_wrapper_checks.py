"""GPU test of the Python wrappers' quick checks: they accept exactly what the checks that name the
fault accept, and a fused call hands over the same segments as hq_segment structures."""
import ctypes

import pytest

from nebula_amd import hq

pytestmark = pytest.mark.gpu


def raises(f, *a):
    try:
        f(*a)
        return False
    except ValueError:
        return True


def test_quick_checks_agree_with_the_named_ones(cuda):
    import torch

    c = lambda *s, dtype=torch.float16: torch.zeros(*s, dtype=dtype, device="cuda")
    X = c(3, 256)
    for t in (X, X[:, :128], X[:2], c(3, 512)[:, ::2], c(256, 3).t(), c(1, 256), c(256), c(3, 256).cpu(), c(3, 256).bfloat16(),
              torch.as_strided(X, (3, 256), (8, 1)), c(3, 1), c(0, 256)):
        for rows, cols in ((3, 256), (1, 128), (2, 1)):
            assert hq._rows_ok(t, rows, cols, torch.float16) != raises(hq._check_rows, "t", t, rows, cols, torch.float16)
    K, N, g = 256, 40, 128
    for fmt in (hq.FORMAT_INT4, hq.FORMAT_TERNARY2):
        w = c(hq.packed_words(fmt, K, N), dtype=torch.int32)
        s, b = c(K // g, N), c(K // g, N, dtype=torch.float32)
        for args in ((w, s, None, K, N, g), (w, s, b, K, N, g), (w[:-1], s, None, K, N, g), (w, s[:1], None, K, N, g),
                     (w.cpu(), s, None, K, N, g), (w, s.cpu(), None, K, N, g), (w, s.float(), None, K, N, g),
                     (w.view(2, -1).t(), s, None, K, N, g), (w, s, b.half(), K, N, g), (w, s, b[:1], K, N, g),
                     (w, s, b.cpu(), K, N, g), (w, s, None, K, N, 96), (w, s, None, K, N, 0), (w, s, None, K, N + 16, g)):
            wp, sc, bias, k, n, grp = args
            assert hq._weight_ok(fmt, *args, X.get_device()) != raises(hq._check_weight, fmt, wp, sc, bias, k, n, grp, X), args[3:]


def test_packed_segments_are_the_structures():
    seg = hq.Segment(0x1122334455667788, 2, None, 4, -5, 6)
    assert hq._SEGMENT.pack(0x1122334455667788, 2, 0, 4, -5, 6) == bytes(seg)
    assert ctypes.sizeof(hq.Segment) == hq._SEGMENT.size
