"""Quantisation paths taken by size: the one-launch cast of small tensors."""
import numpy as np
import pytest
import torch

from oracle import fp8 as ofp8
from oracle import quant as oq
from tcfp_amd import kernels as K

pytestmark = pytest.mark.gpu


def _kernel_names(fn):
    from torch.profiler import ProfilerActivity, profile

    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    return [e.name for e in prof.events()]


# one element, a tail only, one vector, a tail behind the last vector, the
# largest single-workgroup tensor, and the first of two passes
@pytest.mark.parametrize("n", [1, 7, 8, 1027, 32768, 32769])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("fp8", [torch.float8_e4m3fn, torch.float8_e5m2])
def test_small_cast_in_one_launch(dev, n, dtype, fp8):
    x = torch.randn(n, generator=torch.Generator().manual_seed(n)).to(dtype)
    x[n // 2] = -7.25  # the amax, in a tail for the odd sizes
    xd = x.to(dev)
    q, inv, s = K.quantize_per_tensor(xd, fp8, return_scale=True)
    fmt = ofp8.E5M2 if fp8 == torch.float8_e5m2 else ofp8.E4M3
    codes, oinv, oscale = oq.to_fp8_per_tensor(
        x.float().numpy(), "bf16" if dtype == torch.bfloat16 else "f32", fmt)
    assert np.array_equal(q.view(torch.uint8).cpu().numpy(), codes)
    assert inv.item() == float(oinv) and s.item() == float(oscale)
    names = _kernel_names(lambda: K.quantize_per_tensor(xd, fp8))
    assert any("quant_one_kernel" in k for k in names) == (n <= 32768)


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), 0.0])
def test_small_cast_special_values(dev, bad):
    """The codes and the scale of the two-pass form (the same values inside a
    larger tensor of zeros)."""
    x = torch.randn(1000, generator=torch.Generator().manual_seed(1))
    x = torch.zeros(1000) if bad == 0.0 else x
    x[123] = bad
    big = torch.zeros(40000)
    big[:1000] = x
    q, inv = K.quantize_per_tensor(x.to(dev))
    qb, invb = K.quantize_per_tensor(big.to(dev))
    assert torch.equal(q.view(torch.uint8), qb.view(torch.uint8)[:1000])
    assert torch.equal(inv.isnan(), invb.isnan())
    assert torch.equal(inv.nan_to_num(), invb.nan_to_num())
