"""The native host module's boundary, as far as it runs without a GPU: what
its functions accept, and how their errors reach Python."""
import pytest
import torch

from tcfp_amd import kernels as K


@pytest.mark.parametrize("seed", [-1, 0, 2**63, 2**64 + 5, torch.tensor(7)])
def test_dual_quantise_takes_any_integer_seed(seed):
    """The seed counts modulo 2^64; a CPU weight is then refused for its
    device, the first thing the op itself checks."""
    with pytest.raises(RuntimeError, match="only on the GPU"):
        K.dual_quantize_per_tensor(torch.zeros(8, 16), stochastic_lo=True, seed=seed)
