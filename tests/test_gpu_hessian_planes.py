"""The bf16 planes of an fp32 Hessian, value by value: what they do not hold
takes the fp32 product, as the call without a workspace does."""
import ctypes as C

import pytest
import torch

from llmcompressor_amd import _lib as L
from llmcompressor_amd import ops


def _fp32_product(x, alpha=2.0, H=None, beta=0.0):
    """The call without a workspace."""
    n, d = x.shape
    H = torch.zeros(d, d, device=x.device) if H is None else H
    L.check(L.lib().mi355q_hessian_syrk(x.data_ptr(), L.F32, n, d, x.stride(0), H.data_ptr(), d, C.c_float(alpha),
                                        C.c_float(beta), None, 0, L.stream_of(x)))
    return H


def _hessian(x, alpha=2.0):
    d = x.shape[1]
    return ops.hessian_syrk_(torch.zeros(d, d, device=x.device), x, alpha=alpha, beta=0.0)


@pytest.mark.gpu
@pytest.mark.parametrize("value", [1e21, -1e25, 2.3e30, 1.7e38])
def test_products_that_overflow(dev, value):
    """Finite values whose squares overflow: an infinity, as fp32 arithmetic gives, and no NaN."""
    g = torch.Generator(device=dev)
    g.manual_seed(7)
    x = torch.randn(768, 640, generator=g, device=dev)
    # significands that bf16 rounds up and down
    for k in range(64):
        x[8 * k, 9 * k] = value * (1 + k / 64) / 2
    H = torch.triu(_hessian(x))
    assert not torch.isnan(H).any()
    assert bool((torch.diagonal(H)[9 * torch.arange(64)] == float("inf")).all())
    assert torch.equal(H, torch.triu(_fp32_product(x)))
