"""GPU test of the prefill kernels' ternary weights under bf16 activations over every kind of fp16
group scale. One-hot activation rows pick single weights, so each output is the bf16 rounding of
t * s with no sum behind it: the comparison is exact."""
import numpy as np
import pytest

import oracle as O
from gpu_util import DeviceProblem, to_host_f32
from nebula_amd import hq

pytestmark = pytest.mark.gpu


# 64-row, 128-row, 128-column and general (64-row) tiles.
@pytest.mark.parametrize("env", [{"HQ_PREFILL_RT": "4"}, {"HQ_PREFILL_WM": "1", "HQ_PREFILL_KS": "1"},
                                 {"HQ_PREFILL_TW": "2", "HQ_PREFILL_WM": "1"}, {"HQ_GENERAL": "1"}])
def test_ternary_bf16_prefill_scales_exact(cuda, monkeypatch, env):
    M, K, N, group = 300, 384, 600, 128
    P = O.Problem(O.TERNARY2, M, K, N, group, O.BF16, seed=8800)
    bits = np.linspace(0, 0xFFFF, 3 * N).astype(np.uint16)  # zeros, subnormals, normals, Inf, NaN, both signs
    bits[[0, 1, 2, 3, 4, 5, 6]] = [0x0000, 0x8000, 0x0001, 0x03FF, 0x0400, 0x7BFF, 0xFBFF]
    P.scales = np.random.default_rng(1).permutation(bits).reshape(3, N)
    one = np.zeros((M, K), dtype=np.uint16)
    one[np.arange(M), (7 * np.arange(M)) % K] = 0x3F80  # bf16 1.0
    P.X = one
    D = DeviceProblem(P)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    assert "prefill" in hq.describe(P.fmt, O.BF16, M, K, N, group)
    y = to_host_f32(D.run())
    ref = P.reference()  # fp32 t * s (0 for a group without a finite scale)
    import torch

    want = torch.from_numpy(ref).to(torch.bfloat16).float().numpy()
    assert np.array_equal(y, want), np.argwhere(y != want)[:4]
