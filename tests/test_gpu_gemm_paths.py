"""GEMM paths the dispatcher takes by size: the four-stage small tile with
block exponents.

Bounds: 1e-4 relative Frobenius with fp32 output (the FP8 MFMA's internal sum
of a block is a flat ~1.5e-5 off a float64 matmul of the same operands; an
indexing or scaling slip is of order 1), 3e-3 with bf16 output (one rounding
to 8 significant bits: RMS 1.1e-3).
"""
import pytest
import torch

from tcfp_amd import kernels as K

pytestmark = pytest.mark.gpu


def _kernel_names(fn):
    from torch.profiler import ProfilerActivity, profile

    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    return [e.name for e in prof.events()]


def _rel(out, ref):
    return (torch.linalg.norm(out.double() - ref) / torch.linalg.norm(ref)).item()


def _deq(q, e, bs):
    return q.double() * torch.exp2(e.t().double()).repeat_interleave(bs, dim=1)


@pytest.mark.parametrize("bs", [32, 64, 128])
@pytest.mark.parametrize("m,n,k", [(100, 130, 640), (257, 500, 768), (1000, 512, 4096),
                                   (65, 96, 1920)])
def test_four_stage_block_exponents_match_two_stage(dev, m, n, k, bs):
    """The four-stage tile (exponents through LDS) gives the bits of the
    two-stage tile with the same activation codes, which the fused
    activation-quant launch runs, on ragged rows, columns and alignments."""
    g = torch.Generator().manual_seed(m + n + k + bs)
    x = (torch.randn(m, k, generator=g)
         * torch.exp2(torch.randint(-6, 7, (m, k // bs), generator=g)
                      ).repeat_interleave(bs, dim=1)).to(dev)
    w = torch.randn(n, k, generator=g) * torch.exp2(torch.randint(-9, 9, (n, 1), generator=g))
    hi, lo, eh, el = K.fused_dual_quantize_fp8(w.to(dev), bs)
    a, ea = K.block_quantize_fp8(x, bs)
    names = _kernel_names(lambda: K.fused_block_scaled_dual_gemm_forward(a, hi, lo, ea, eh, el, bs))
    assert any("4, 128, 64, 1, 4, 0, 0>" in s for s in names), names
    out = K.fused_block_scaled_dual_gemm_forward(a, hi, lo, ea, eh, el, bs)
    fused, _, _ = K.fused_act_quant_dual_gemm_forward(x, hi, lo, eh, el, bs)
    assert torch.equal(out, fused)
    ref = _deq(a, ea, bs) @ (_deq(hi, eh, bs) + _deq(lo, el, bs)).t()
    assert _rel(out, ref) < 1e-4
    single = K.block_scaled_gemm(a, hi, ea, eh, bs)
    assert _rel(single, _deq(a, ea, bs) @ _deq(hi, eh, bs).t()) < 1e-4
