"""GEMM paths the dispatcher takes by size: the weight stream for few
activation rows, and the four-stage small tile with block exponents.

Bounds: 1e-4 relative Frobenius with fp32 output (the FP8 MFMA's internal sum
of a block is a flat ~1.5e-5 off a float64 matmul of the same operands; an
indexing or scaling slip is of order 1), 3e-3 with bf16 output (one rounding
to 8 significant bits: RMS 1.1e-3).
"""
import pytest
import torch

from tcfp_amd import kernels as K

pytestmark = pytest.mark.gpu

E4M3, E5M2 = torch.float8_e4m3fn, torch.float8_e5m2


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


# rows at the edges of the 16 / 32 / 64-row variants, columns at those of the
# 16-column workgroups and of the rule (N <= 8192 up to 32 rows, else 2048),
# contractions with a partial last 128-column step (K % 16 == 0), fewer steps
# than waves, and steps that the eight waves share unevenly
FEW = [(1, 16, 16), (1, 1024, 1024), (16, 8192, 4096), (17, 130, 1040), (32, 8192, 272),
       (33, 2048, 80), (48, 1001, 4096), (64, 2048, 1168), (64, 513, 128)]


@pytest.mark.parametrize("dual", [True, False])
@pytest.mark.parametrize("fmt", [E4M3, E5M2])
@pytest.mark.parametrize("m,n,k", FEW)
def test_few_rows_per_tensor(dev, m, n, k, fmt, dual):
    g = torch.Generator().manual_seed(m * 7 + n + k)
    a, sa = K.quantize_per_tensor(torch.randn(m, k, generator=g).to(dev), fmt)
    hi, lo, ih, il = K.dual_quantize_per_tensor(torch.randn(n, k, generator=g).to(dev))
    bias = torch.randn(n, generator=g).to(dev)
    ref = (a.double() * sa.double()) @ (
        hi.double() * ih.double() + (lo.double() * il.double() if dual else 0)).t() + bias.double()
    for od, tol in ((torch.float32, 1e-4), (torch.bfloat16, 3e-3)):
        def run():
            if dual:
                return K.fused_dual_gemm_forward(a, hi, lo, sa, ih, il, bias=bias, out_dtype=od)
            return K.fp8_gemm_nt(a, hi, sa, ih, bias=bias, out_dtype=od)

        out = run()
        assert any("gemm_skinny" in x for x in _kernel_names(run))
        err = _rel(out, ref)
        print(f"few rows {m}x{n}x{k} {od} dual={dual} rel_fro {err:.2e}")
        assert err < tol
        assert torch.equal(out, run())  # the waves' sums meet in a fixed order


@pytest.mark.parametrize("bs", [32, 64, 128])
@pytest.mark.parametrize("dual", [True, False])
@pytest.mark.parametrize("m,n,kb", [(1, 1024, 1), (16, 8192, 9), (17, 520, 5), (33, 1001, 17),
                                    (64, 2048, 32)])
def test_few_rows_block_exponents(dev, m, n, kb, bs, dual):
    """Per-column scales spread over many binades, so that an exponent taken
    from another block or row is an error of order 1."""
    k = kb * bs
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g) * torch.exp2(torch.randint(-6, 7, (m, k), generator=g))
    w = torch.randn(n, k, generator=g) * torch.exp2(torch.randint(-6, 7, (n, k), generator=g))
    a, ea = K.block_quantize_fp8(x.to(dev), bs)
    hi, lo, eh, el = K.fused_dual_quantize_fp8(w.to(dev), bs)
    ref = _deq(hi, eh, bs)
    if dual:
        ref = ref + _deq(lo, torch.where(el == -128, torch.full_like(el, -127), el), bs)
    ref = _deq(a, ea, bs) @ ref.t()
    for od, tol in ((torch.float32, 1e-4), (torch.bfloat16, 3e-3)):
        def run():
            if dual:
                return K.fused_block_scaled_dual_gemm_forward(a, hi, lo, ea, eh, el, bs,
                                                              out_dtype=od)
            return K.block_scaled_gemm(a, hi, ea, eh, bs, out_dtype=od)

        out = run()
        assert any("gemm_skinny" in x for x in _kernel_names(run))
        err = _rel(out, ref)
        print(f"few rows {m}x{n}x{k} bs {bs} {od} dual={dual} rel_fro {err:.2e}")
        assert err < tol


# both sides of the weight stream's lines: 17 to 32 rows and more output columns
# than CUs x 16, where it pays for short contractions only
@pytest.mark.parametrize("m,n,k,bs,stream", [
    (17, 4096, 1040, 0, True), (32, 4112, 512, 0, True), (17, 4112, 528, 0, False),
    (32, 8192, 4096, 0, False), (17, 4112, 2048, 64, True), (32, 8192, 2176, 128, False)])
def test_few_rows_of_wide_weights(dev, m, n, k, bs, stream):
    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn(m, k, generator=g).to(dev), torch.randn(n, k, generator=g).to(dev)
    if bs:
        a, ea = K.block_quantize_fp8(x, bs)
        hi, lo, eh, el = K.fused_dual_quantize_fp8(w, bs)
        ref = _deq(a, ea, bs) @ (_deq(hi, eh, bs) + _deq(lo, el, bs)).t()

        def run():
            return K.fused_block_scaled_dual_gemm_forward(a, hi, lo, ea, eh, el, bs)
    else:
        a, sa = K.quantize_per_tensor(x)
        hi, lo, ih, il = K.dual_quantize_per_tensor(w)
        ref = (a.double() * sa.double()) @ (hi.double() * ih.double()
                                            + lo.double() * il.double()).t()

        def run():
            return K.fused_dual_gemm_forward(a, hi, lo, sa, ih, il)
    assert any("gemm_skinny" in x for x in _kernel_names(run)) == stream
    assert _rel(run(), ref) < 1e-4


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


# the 128 x 128 tile: full and partial tiles on both sides, a partial last
# stage (K % 128 != 0), fewer stages than buffers under the forcing policy,
# and the shapes the rule sends there
MID = [("auto", 1000, 4096, 1040, 0), ("auto", 2048, 2048, 1024, 64), ("auto", 600, 4000, 2048, 32),
       ("auto", 600, 4000, 2048, 128), ("mid", 130, 200, 16, 0), ("mid", 1, 129, 272, 0),
       ("mid", 257, 250, 64, 64), ("mid", 100, 385, 96, 32), ("mid", 128, 128, 384, 128)]


@pytest.mark.parametrize("od", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("policy,m,n,k,bs", MID)
def test_mid_tile_matches_small_tile(dev, policy, m, n, k, bs, od):
    """The 128 x 128 tile's bits are the 128 x 64 tile's (the same products in
    the same order of K), with a bias, and within the bound of float64."""
    g = torch.Generator().manual_seed(m + n + k + bs)
    x = torch.randn(m, k, generator=g).to(dev)
    w = (torch.randn(n, k, generator=g)
         * torch.exp2(torch.randint(-9, 9, (n, 1), generator=g))).to(dev)
    bias = torch.randn(n, generator=g).to(dev)
    if bs:
        a, ea = K.block_quantize_fp8(x, bs, E5M2)
        hi, lo, eh, el = K.fused_dual_quantize_fp8(w, bs)
        ref = _deq(a, ea, bs) @ (_deq(hi, eh, bs) + _deq(lo, el, bs)).t()

        def run():
            return K.fused_block_scaled_dual_gemm_forward(a, hi, lo, ea, eh, el, bs, bias=bias,
                                                          out_dtype=od)
    else:
        a, sa = K.quantize_per_tensor(x, E5M2)
        hi, lo, ih, il = K.dual_quantize_per_tensor(w)
        ref = (a.double() * sa.double()) @ (hi.double() * ih.double()
                                            + lo.double() * il.double()).t()

        def run():
            return K.fused_dual_gemm_forward(a, hi, lo, sa, ih, il, bias=bias, out_dtype=od)
    try:
        K.set_gemm_tile_policy("small")
        small = run()
        K.set_gemm_tile_policy(policy)
        names = _kernel_names(run)
        out = run()
    finally:
        K.set_gemm_tile_policy("auto")
    assert any("4, 128, 128, " in s for s in names), names
    assert torch.equal(out, small)
    assert _rel(out, ref + bias.double()) < (1e-4 if od == torch.float32 else 3e-3)


@pytest.mark.parametrize("m,n,k,mid", [(1000, 4096, 1024, False), (1000, 4096, 1536, True),
                                       (600, 4096, 1104, True), (500, 8192, 1408, False)])
def test_mid_tile_one_round_line(dev, m, n, k, mid):
    """Per tensor, in one round of the 128 x 128 tile: K from 1536 on, from 1024
    where the operand rows do not start on 128-byte lines."""
    g = torch.Generator().manual_seed(k)
    a, sa = K.quantize_per_tensor(torch.randn(m, k, generator=g).to(dev))
    hi, lo, ih, il = K.dual_quantize_per_tensor(torch.randn(n, k, generator=g).to(dev))
    ref = (a.double() * sa.double()) @ (hi.double() * ih.double() + lo.double() * il.double()).t()

    def run():
        return K.fused_dual_gemm_forward(a, hi, lo, sa, ih, il)
    assert any("4, 128, 128, " in s for s in _kernel_names(run)) == mid
    assert _rel(run(), ref) < 1e-4


# every tile a dgrad may take: the weight stream, one round of the small tile,
# the 128 x 128 tile, the large one, the persistent one with eight and four waves
@pytest.mark.parametrize("m,n,k", [(40, 520, 256), (300, 512, 400), (1000, 4096, 1024),
                                   (1000, 4096, 1552), (8192, 1024, 384), (4096, 4096, 256), (2048, 4608, 8192)])
def test_bf16_gradient_is_the_rounded_fp32_one(dev, m, n, k):
    g = torch.Generator().manual_seed(m + k)
    a, sa = K.quantize_per_tensor(torch.randn(m, k, generator=g).to(dev), E5M2)
    hi, lo, ih, il = K.dual_quantize_per_tensor(torch.randn(n, k, generator=g).to(dev))
    f32 = K._dual_gemm(a, hi, lo, sa, ih, il, None, torch.float32)
    assert torch.equal(K._dual_gemm(a, hi, lo, sa, ih, il, None, torch.bfloat16), f32.bfloat16())


@pytest.mark.parametrize("m,n,k", [(100, 128, 192), (4096, 256, 1024), (2048, 4096, 8192),
                                   (4096, 2048, 4096)])
def test_block_backward_bf16_gradient(dev, m, n, k):
    """block_linear_backward's dX in bf16 is its fp32 dX rounded (with W_lo, and
    W_hi alone), dW and db the same."""
    g = torch.Generator().manual_seed(m + k)
    gr = torch.randn(m, n, generator=g).to(dev)
    out = K.block_linear_forward(torch.randn(m, k, generator=g).bfloat16().to(dev),
                                 (torch.randn(n, k, generator=g) * 0.02).to(dev), None, 64)
    _, hi, lo, eh, el, aq, ae = out
    for lo_, el_ in ((lo, el), (None, None)):
        ref = K.block_linear_backward(gr, aq, ae, hi, lo_, eh, el_, 64, True, True, True)
        got = K.block_linear_backward(gr, aq, ae, hi, lo_, eh, el_, 64, True, True, True,
                                      dx_dtype=torch.bfloat16)
        assert torch.equal(got[0], ref[0].bfloat16())
        assert torch.equal(got[1], ref[1]) and torch.equal(got[2], ref[2])


# more 256 x 128 tiles than CUs with partial tiles at the right, below and
# both, a partial last stage (K % 128 != 0) and none, tile counts that the
# eight XCDs share unevenly, outputs narrower than a tile, exponent chunks
# outside the matrix and exponent blocks past K
RAGGED = [(4097, 4104, 144, 0), (4000, 4352, 1024, 0), (4096, 4096 + 8, 400, 0),
          (65793, 8, 272, 0), (260, 17000, 400, 0), (4112, 4112, 288, 32), (4352, 4112, 320, 64),
          (65552, 16, 384, 128), (4336, 4096, 416, 32)]


@pytest.mark.parametrize("od", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k,bs", RAGGED)
def test_ragged_persistent_tiles_match_small_tile(dev, m, n, k, bs, od):
    """Back-to-back tiles of ragged matrices give the bits of the 128 x 64
    tile (the same products in the same order of K), with and without a bias."""
    g = torch.Generator().manual_seed(m + n + k + bs)
    x = torch.randn(m, k, generator=g).to(dev)
    w = (torch.randn(n, k, generator=g)
         * torch.exp2(torch.randint(-9, 9, (n, 1), generator=g))).to(dev)
    for bias in (None, torch.randn(n, generator=g).to(dev)):
        if bs:
            a, ea = K.block_quantize_fp8(x, bs, E5M2)
            hi, lo, eh, el = K.fused_dual_quantize_fp8(w, bs)

            def run():
                return K.fused_block_scaled_dual_gemm_forward(a, hi, lo, ea, eh, el, bs,
                                                              bias=bias, out_dtype=od)
        else:
            a, sa = K.quantize_per_tensor(x)
            hi, lo, ih, il = K.dual_quantize_per_tensor(w)

            def run():
                return K.fused_dual_gemm_forward(a, hi, lo, sa, ih, il, bias=bias, out_dtype=od)
        names = _kernel_names(run)
        assert any("gemm_nt_ragged_kernel" in s for s in names), names
        out = run()
        try:
            K.set_gemm_tile_policy("small")
            assert torch.equal(out, run())
        finally:
            K.set_gemm_tile_policy("auto")
