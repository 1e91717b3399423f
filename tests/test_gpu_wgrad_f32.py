"""The weight gradient of token counts that the FP8 and the split-bf16 products
do not take: G^T deq(X) in fp32 accuracy as three exact bf16 passes.

Bound: the fp32 product's own error.  The split is exact, so what is left is
fp32 accumulation over the tokens: at most (3 m / 16 + a few) roundings of
2^-24 per element, random in sign, against m for an fp32 dot; the test holds
the relative Frobenius error to 1.2 times torch's fp32 product of the same
operands or 2e-7, whichever is larger (2^-24 = 6e-8 is one rounding)."""
import pytest
import torch

from tcfp_amd import kernels as K
from tcfp_amd.nn import TCFPLinear

pytestmark = pytest.mark.gpu


def _rel(out, ref):
    return (torch.linalg.norm(out.double() - ref) / torch.linalg.norm(ref)).item()


# one token, the edges of the 64-row padding, ragged columns, split-K and more
# than one chunk of dW rows (64 MiB of split gradient: m 2001 x n 6000)
@pytest.mark.parametrize("m,n,k", [(1, 16, 16), (63, 130, 80), (65, 48, 1040), (1000, 1552, 1040),
                                   (1001, 33, 4096), (2001, 6000, 272)])
@pytest.mark.parametrize("fp8", [torch.float8_e4m3fn, torch.float8_e5m2])
def test_per_tensor(dev, m, n, k, fp8):
    gen = torch.Generator().manual_seed(m + n)
    g = (torch.randn(m, n, generator=gen)
         * torch.exp2(torch.randint(-20, 20, (1, n), generator=gen))).to(dev)
    q, inv = K.quantize_per_tensor(torch.randn(m, k, generator=gen).to(dev), fp8)
    dw = K.wgrad_f32(g, q, inv)
    # (per column scale of g: errors are compared row by row of dW)
    ref = g.double().t() @ (q.double() * inv.double())
    s = ref.norm(dim=1, keepdim=True).clamp(min=1e-300)
    fp32 = g.t() @ (q.float() * inv)
    err, own = _rel(dw / s, ref / s), _rel(fp32 / s, ref / s)
    print(f"wgrad_f32 {m}x{n}x{k} {fp8}: {err:.2e} (torch fp32 {own:.2e})")
    assert err <= max(1.2 * own, 2e-7)
    assert torch.equal(dw, K.wgrad_f32(g, q, inv))


@pytest.mark.parametrize("bs", [32, 64, 128])
@pytest.mark.parametrize("m", [1, 101, 1027])
def test_block(dev, m, bs):
    n, k = 200, 512
    gen = torch.Generator().manual_seed(m + bs)
    g = torch.randn(m, n, generator=gen).to(dev)
    x = torch.randn(m, k, generator=gen) * torch.exp2(torch.randint(-8, 8, (m, k), generator=gen))
    q, e = K.block_quantize_fp8(x.to(dev), bs)
    dw = K.block_scaled_wgrad(g, q, e, bs)
    xd = K.block_dequantize_fp8(q, e, bs)
    ref = g.double().t() @ xd.double()
    assert _rel(dw, ref) <= max(1.2 * _rel(g.t() @ xd, ref), 2e-7)


def _same(x, ref):
    """Equal values, NaN equal to NaN, an inf only to the same inf."""
    return torch.equal(x.isnan(), ref.isnan()) and torch.equal(
        torch.where(x.isnan(), 0, x), torch.where(ref.isnan(), 0, ref))


def test_special_gradients(dev):
    """Non-finite and extreme gradients as the fp32 product has them: an inf
    row stays inf, a NaN NaN, the largest and smallest normals are exact."""
    m, n, k = 19, 64, 32
    q = torch.ones(m, k, device=dev).to(torch.float8_e4m3fn)
    inv = torch.ones(1, device=dev)
    g = torch.zeros(m, n, device=dev)
    g[3, 0] = float("inf")
    g[4, 1] = float("nan")
    g[5, 2] = torch.finfo(torch.float32).max
    g[6, 3] = -1.2345678e-20
    g[7, 4] = float("-inf")
    g[8, 5] = torch.finfo(torch.float32).tiny
    dw = K.wgrad_f32(g, q, inv)
    assert _same(dw, g.t() @ q.float())


@pytest.mark.parametrize("inv", [0.0123, 2.0**-60, 1.7e-38, 3.0, 5e8, float("nan")])
@pytest.mark.parametrize("fp8", [torch.float8_e4m3fn, torch.float8_e5m2])
def test_scale_ahead_of_the_sum(dev, inv, fp8):
    """Gradients whose products with the codes pass fp32's range where those
    with the scaled codes do not, and the reverse: finite where the fp32
    product is, to the same accuracy."""
    m, n, k = 35, 48, 64
    gen = torch.Generator().manual_seed(7)
    q = (torch.randn(m, k, generator=gen) * 100).to(fp8).to(dev)
    s = torch.full((1,), inv, device=dev)
    # (products up to 2e36 * 4 * 400 > 3.4e38; results of 35 terms of deviation 2e36 *
    # 100 * 0.0123 stay ten deviations, 1.5e37 each, inside the range, whatever the order)
    mag = 2e36 if inv < 1 else 1e30 / inv
    g = (torch.randn(m, n, generator=gen) * mag).to(dev)
    dw, ref = K.wgrad_f32(g, q, s), g.double().t() @ (q.double() * s.double())
    fp32 = g.t() @ (q.float() * s)
    assert torch.equal(dw.isfinite(), fp32.isfinite())
    if fp32.isfinite().any():
        assert _rel(dw, ref) <= max(1.2 * _rel(fp32, ref), 2e-7)


def test_layer_uses_it(dev):
    """A per-tensor layer's dW at 1000 tokens against 64 bits."""
    torch.manual_seed(0)
    layer = TCFPLinear(256, 320, use_tensor_cores=True).to(dev)
    x = torch.randn(1000, 256, device=dev)
    g = torch.randn(1000, 320, device=dev)
    layer(x).backward(g)
    q, inv = K.quantize_per_tensor(x)
    ref = g.double().t() @ (q.double() * inv.double())
    assert _rel(layer.weight.grad, ref) < 1e-6


@pytest.mark.parametrize("bs", [0, 32])
def test_millions_of_tokens(dev, bs):
    """More tokens than one launch's descriptors span (2.8 million at the 128-row
    tile), an odd number of them."""
    m, n, k = 2_900_003, 16, 32
    gen = torch.Generator(device=dev).manual_seed(3)
    g = torch.randn(m, n, generator=gen, device=dev)
    x = torch.randn(m, k, generator=gen, device=dev)
    if bs:
        q, e = K.block_quantize_fp8(x, bs)
        dw, deq = K.block_scaled_wgrad(g, q, e, bs), K.block_dequantize_fp8(q, e, bs)
    else:
        q, inv = K.quantize_per_tensor(x)
        dw, deq = K.wgrad_f32(g, q, inv), q.float() * inv
    ref = g.double().t() @ deq.double()
    # (sums of 2.9e6 terms that cancel to 1.7e3: the fp32 product's own error)
    assert _rel(dw, ref) <= max(1.2 * _rel(g.t() @ deq, ref), 2e-7)


@pytest.mark.parametrize("bs", [None, 32])
def test_layer_under_create_graph(dev, bs):
    """A gradient penalty on dW at an odd token count: the weight gradient of a
    frozen input is linear in the output's gradient and can be differentiated.
    With A the dequantised activation, out's gradient 2 out and s = sum dW^2:
    ds/dout = 4 A dW^T, and ds/dW = (4 A dW^T)^T A."""
    torch.manual_seed(0)
    m = 35
    layer = TCFPLinear(64, 96, use_tensor_cores=True, scale_block_size=bs, bias=False,
                       error_feedback=False).to(dev)
    x = torch.randn(m, 64, device=dev)
    out = layer(x)
    dw, = torch.autograd.grad(out.square().sum(), layer.weight, create_graph=True)
    got, = torch.autograd.grad(dw.square().sum(), layer.weight)
    a = (K.block_dequantize_fp8(*K.block_quantize_fp8(x, bs), bs) if bs else
         K.quantize_per_tensor(x)[0].float() * K.quantize_per_tensor(x)[1]).double()
    ref = (2 * out.detach().double()).t() @ a
    assert _rel(dw, ref) < 1e-6
    assert _rel(got, (4 * a @ ref.t()).t() @ a) < 1e-6


@pytest.mark.parametrize("bs", [None, 32])
def test_layer_with_batched_gradients(dev, bs):
    torch.manual_seed(0)
    m = 35
    layer = TCFPLinear(64, 96, use_tensor_cores=True, scale_block_size=bs, bias=False,
                       error_feedback=False).to(dev)
    out = layer(torch.randn(m, 64, device=dev))
    gs = torch.randn(3, m, 96, device=dev)
    batched, = torch.autograd.grad(out, layer.weight, gs, retain_graph=True, is_grads_batched=True)
    each = [torch.autograd.grad(out, layer.weight, g, retain_graph=True)[0] for g in gs]
    mapped = torch.func.vmap(
        lambda g: torch.autograd.grad(out, layer.weight, g, retain_graph=True)[0])(gs)
    for b in (batched, mapped):
        assert _rel(b, torch.stack(each).double()) < 1e-6
