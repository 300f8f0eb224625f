"""fp32 activations on the 16-bit matrix kernel: three bf16 planes per value.

From 512 rows and 512 columns on an fp32 Hessian is summed from six plane
products; below, and for values that the planes do not hold (infinities, NaN,
magnitudes of 2^54 and above, nonzero ones below 2^-110), by the fp32 product.
The split is exact (24 bits of significand in three times 8) and the dropped terms are
below 2^-24 of each product, so the error against float64 is that of an fp32
sum of n products: at most n roundings of a partial sum, i.e. n 2^-24 of sum
|x_i x_j|, which is at most the product of the two columns' norms.
"""
import pytest
import torch

from llmcompressor_amd import ops

pytestmark = pytest.mark.gpu

ULP = 2.0 ** -24


def _rows(n, d, dev, seed):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    c = torch.exp(3 * torch.randn(d, generator=g, device=dev))
    return torch.randn(n, d, generator=g, device=dev) * c


def _f64(x, alpha, H0, beta):
    x = x.double()
    return torch.triu(beta * H0.double() + alpha * (x.t() @ x))


# both sides of the 512 lines; rows off the 128-row chunks; widths off every
# vector size and tile; several calls of planes would need 1 GiB: not here
@pytest.mark.parametrize("n,d", [(511, 512), (512, 511), (512, 512), (513, 513), (640, 1001), (2049, 770),
                                 (4096, 1024), (700, 2056)])
@pytest.mark.parametrize("beta", [0.0, 0.5, 1.0])
def test_against_f64(dev, n, d, beta):
    x = _rows(n, d + 5, dev, n + d)[:, 2:2 + d]     # a row stride of its own, unaligned rows
    H0 = torch.randn(d, d, device=dev)
    H = H0.clone()
    ops.hessian_syrk_(H, x, alpha=2.0, beta=beta)
    assert torch.equal(torch.tril(H, -1), torch.tril(H0, -1))     # the lower triangle is left alone
    want = _f64(x, 2.0, H0, beta)
    got = torch.triu(H).double()
    scale = torch.sqrt(torch.outer(torch.diagonal(_f64(x, 2.0, H0 * 0, 0.0)), torch.diagonal(
        _f64(x, 2.0, H0 * 0, 0.0)))) + H0.abs().double()
    # n roundings, and those of beta H, of the sum and of alpha
    assert float(((got - want).abs() / scale).max()) <= (n + 3) * ULP
    H2 = H0.clone()
    ops.hessian_syrk_(H2, x, alpha=2.0, beta=beta)
    assert torch.equal(H, H2)


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4e38, -float("inf")])
def test_values_the_planes_do_not_hold(dev, value):
    """The fp32 product takes the call: finite columns keep their sums, and
    an infinity meets the infinities and NaNs that fp32 arithmetic gives."""
    n, d = 768, 640
    x = _rows(n, d, dev, 5)
    x[5, 7] = value
    x[5, 9] = 0.0
    H = torch.zeros(d, d, device=dev)
    ops.hessian_syrk_(H, x, alpha=2.0, beta=0.0)
    keep = [i for i in range(d) if i != 7]
    got, want = H[keep][:, keep].double(), _f64(x[:, keep], 2.0, torch.zeros(d - 1, d - 1, device=dev), 0.0)
    assert float(torch.linalg.norm(torch.triu(got) - want) / torch.linalg.norm(want)) <= 1e-6
    assert bool(torch.isnan(H[7, 9])) == (value != 3.4e38)
    assert not torch.isfinite(H[7, 7])


def test_small_values_keep_their_columns(dev):
    """Columns of very different sizes (1e-18 .. 1e17: the sums stay below fp32 overflow) keep their own precision
    (values of 2^54 and above among them: the fp32 product takes the call)."""
    n, d = 1024, 512
    x = torch.randn(n, d, device=dev) * torch.logspace(-18, 17, d, device=dev)
    H = torch.zeros(d, d, device=dev)
    ops.hessian_syrk_(H, x, alpha=2.0, beta=0.0)
    want = _f64(x, 2.0, torch.zeros(d, d, device=dev), 0.0)
    s = torch.sqrt(torch.diagonal(want))
    ok = torch.triu(torch.outer(s, s) > 1e-30)     # above the fp32 underflow of the sums
    err = (torch.triu(H).double() - want).abs() / torch.outer(s, s)
    assert float(err[ok].max()) <= (n + 3) * ULP
