"""The bound behind the candidate windows of the per-tensor dual quantisation
(quant.hip, amax_cand_kernel / cand_decisive), evaluated on the CPU: whatever
a filtered round leaves out has a smaller residual than the bound the
decision uses."""
import numpy as np
import pytest

from oracle import fp8 as ofp8

F32 = np.float32
WIN = F32(2.0)


@pytest.mark.parametrize("amax", [F32(0.0311), F32(1.0), F32(437.5), F32(3e-20)])
@pytest.mark.parametrize("short", [0.0, 1e-6, 1e-3, 4e-3])
def test_left_out_values_stay_below_the_bound(amax, short):
    """Every value a filter at M = amax (1 - short) drops, over a dense grid of
    the top binade and the edges of every window."""
    m = F32(amax * F32(1.0 - short))
    s = F32(F32(F32(1.0) / amax) * F32(448.0))
    inv = F32(F32(1.0) / s)
    x = np.linspace(250.0, 448.0, 200_001)
    for mid in range(272, 433, 32):
        x = np.concatenate([x, mid + np.linspace(-2.5, 2.5, 20_001)])
    v = (x / 448.0 * float(m)).astype(F32)
    v = v[v <= m]
    u = np.abs(v) * F32(F32(448.0 / 32.0) / m) - F32(8.5)
    kept = np.abs(u - np.rint(u)) <= WIN / F32(32.0)
    codes = ofp8.encode(np.clip(v * s, F32(-448), F32(448)).astype(F32), ofp8.E4M3)
    res = np.abs(v - (ofp8.decode(codes, ofp8.E4M3).astype(F32) * inv).astype(F32))
    left = max(F32(448.0) * (F32(1.0) - m / amax), F32(0.0))
    bound = max(F32(16.0) - WIN + F32(0.01) + left, F32(8.001)) * inv
    assert (~kept).any() and kept.any()
    assert res[~kept].max() <= bound
    if short <= 1e-3:  # and the windows hold the values that exceed it
        assert res[kept].max() > bound
