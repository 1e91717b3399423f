"""Quantisation paths taken by size and by the data: the one-launch cast of
small tensors, the candidate windows of flat weight distributions, and the
layers' forward without autograd."""
import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as fwAD

from oracle import fp8 as ofp8
from oracle import quant as oq
from tcfp_amd import kernels as K
from tcfp_amd.nn import TCFPLinear, fuse_tcfp_mlp

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


def _flat_case(name, shape, g):
    w = torch.rand(shape, generator=g) * 2 - 1
    if name == "rows":          # every row its own range: most maxima far below the amax
        w = w * (0.6 + 0.4 * torch.rand(shape[0], 1, generator=g))
    elif name == "late":        # the amax comes last, 2% above all before it
        w = w * 0.98
        w[-1, -1] = 1.0
    elif name == "one_short":   # a tenth of a percent above: the windows still decide
        w = w * 0.999
        w[0, 0] = -1.0
    elif name == "edges":       # values on the codes and the midpoints only
        w = (256 + 16 * torch.randint(0, 13, shape, generator=g)).float() / 448
    return w


@pytest.mark.parametrize("name", ["uniform", "rows", "late", "one_short", "edges"])
@pytest.mark.parametrize("wdtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("ef", [True, False])
def test_candidate_windows_match_full_pass(dev, name, wdtype, ef):
    """Flat distributions (the layers' initialisation) keep only the values near
    a midpoint between codes; the results are the full pass's bit for bit,
    where the windows decide and where the maxima lie too far apart."""
    shape = (4096, 2056)
    g = torch.Generator().manual_seed(len(name))
    w = (_flat_case(name, shape, g) * 0.03).to(wdtype).to(dev)
    e = (torch.randn(shape, generator=g) * 1e-6).to(dev) if ef else None
    outs = []
    try:
        for on in (True, False):
            K.set_dual_quant_candidates(on)
            buf = e.clone() if ef else None
            res = K.dual_quantize_per_tensor(w, buf, transposed=True)
            outs.append([r.view(torch.uint8) if r.dtype.itemsize == 1 else r for r in res]
                        + ([buf] if ef else []))
    finally:
        K.set_dual_quant_candidates(True)
    for x, y in zip(*outs):
        assert torch.equal(x, y)


def _requests(monkeypatch, name, pick):
    """What the layers ask of the op `name` from here on, by `pick`."""
    seen, op = [], getattr(K, name)

    def wrapped(*args, **kw):
        seen.append(pick(*args, **kw))
        return op(*args, **kw)

    monkeypatch.setattr(K, name, wrapped)
    return seen


def _batch_copies(dual=(), act=()):
    """(weights' transposed codes, activations' transposed codes) of a batch"""
    return [t for *_, t in dual], [t for *_, t in act]


def test_batched_layer_asks_for_backward_copies_only_when_recording(dev, monkeypatch):
    seen = _requests(monkeypatch, "quantize_batch", _batch_copies)
    layer = TCFPLinear(256, 256, use_tensor_cores=True).to(dev)
    x = torch.randn(48, 256, device=dev, requires_grad=True)
    layer(x)
    with torch.no_grad():
        layer(x)
    assert seen == [([True], [True]), ([False], [False])]


def test_mlp_asks_for_backward_copies_only_when_recording(dev, monkeypatch):
    seen = _requests(monkeypatch, "quantize_batch", _batch_copies)
    gelu = _requests(monkeypatch, "dual_gemm_gelu_quantize",
                     lambda *a, transpose=False, return_dgelu=False, **kw: (transpose,
                                                                            return_dgelu))
    mlp = fuse_tcfp_mlp(torch.nn.Sequential(
        TCFPLinear(256, 512, use_tensor_cores=True), torch.nn.GELU(),
        TCFPLinear(512, 256, use_tensor_cores=True))).to(dev)
    x = torch.randn(64, 256, device=dev, requires_grad=True)
    mlp(x)
    with torch.no_grad():
        mlp(x)
    assert gelu == [(True, True), (False, False)]
    half = len(seen) // 2
    assert all(all(w) and all(a) for w, a in seen[:half])
    assert not any(any(w) or any(a) for w, a in seen[half:])


@pytest.mark.parametrize("kw,d", [({}, 256), ({"scale_block_size": 64}, 1024), ({}, 2944)])
def test_forward_without_autograd_makes_no_backward_copies(dev, kw, d):
    """Under no_grad: the values of the recording forward, no transposed codes
    (by kernel name at d = 2944, the weight beyond the batch's size, where a
    kernel of its own writes them; the batch's are checked above), parameters
    untouched, and forward-mode AD still refused."""
    torch.manual_seed(0)
    layer = TCFPLinear(d, d, use_tensor_cores=True, **kw).to(dev)
    x = torch.randn(48, d, device=dev, requires_grad=True)
    ref = layer(x)
    layer._last_weight_version = -1  # the EF buffer the recording forward wrote
    layer._error_state.reset()
    with torch.no_grad():
        out = layer(x)
        names = _kernel_names(lambda: layer(x))
    assert torch.equal(out, ref.detach()) and not out.requires_grad
    assert not any("dualq_lo_t" in k for k in names)
    assert layer.weight.requires_grad and x.requires_grad
    with torch.no_grad(), fwAD.dual_level(), pytest.raises(RuntimeError):
        layer(fwAD.make_dual(x.detach(), torch.ones_like(x)))


def test_mlp_without_autograd(dev):
    torch.manual_seed(0)
    mlp = fuse_tcfp_mlp(torch.nn.Sequential(
        TCFPLinear(256, 512, use_tensor_cores=True), torch.nn.GELU(),
        TCFPLinear(512, 256, use_tensor_cores=True))).to(dev)
    x = torch.randn(64, 256, device=dev)
    ref = mlp(x)
    for m in (mlp[0], mlp[2]):
        m._error_state.reset()
    with torch.no_grad():
        out = mlp(x)
    assert torch.equal(out, ref.detach()) and not out.requires_grad


def test_out_of_memory_is_torchs_own_error(dev):
    # 4 TiB once contiguous: the allocator refuses it
    x = torch.zeros(1, 1, device=dev).expand(2**20, 2**20)
    with pytest.raises(torch.OutOfMemoryError):
        K.block_quantize_fp8(x, 64)
    assert K.block_quantize_fp8(x[:8, :64], 64)[0].shape == (8, 64)
