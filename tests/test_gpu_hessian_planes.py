"""The bf16 planes of an fp32 Hessian, value by value: what they do not hold
takes the fp32 product, as the call without a workspace does, and what they do
is no further from 64 bits than that product.

Columns that share one token and no other give sums of a single product v w,
so what each of the six plane products carries can be seen.  With h = bf16(v),
m = bf16(v - h), l = v - h - m (|m| <= 2^-8 |v|, |l| <= 2^-17 |v|) the three
products left out, m l', l m' and l l', are together below 1.01 2^-24 |v w|, and
five additions to the first product, which is exact, round by at most 2^-24 of
the sum each: 6.1 2^-24 in all, and the factor of 2 is exact.  h l', l h' or m m'
left out is an error of up to 2^-17.  Each omission breaks the bound on these
inputs (checked below, on the CPU).
"""
import ctypes as C

import pytest
import torch

from llmcompressor_amd import _lib as L
from llmcompressor_amd import ops


ULP = 2.0 ** -24
ONE_PRODUCT = 6.1 * ULP
PAIRS = ((0, 0), (0, 1), (1, 0), (0, 2), (2, 0), (1, 1))


def _single_products(n, d, seed, scale=None):
    """[n, d] with one nonzero value per column, 32 or fewer columns to a
    token, the tokens spread over all rows; full 24-bit significands."""
    g = torch.Generator()
    g.manual_seed(seed)
    v = 1 + torch.rand(d, generator=g)
    v = torch.where(torch.rand(d, generator=g) < 0.5, -v, v)
    if scale is not None:
        v = v * scale
    tokens = torch.randperm(n, generator=g)[: (d + 31) // 32]
    x = torch.zeros(n, d)
    x[tokens[torch.arange(d) % len(tokens)], torch.arange(d)] = v
    return x


def _planes(v):
    h = v.bfloat16().float()
    m = (v - h).bfloat16().float()
    return h.double(), m.double(), (v - h - m).bfloat16().double()


def _error(got, x, alpha=2.0):
    """Largest error of an upper triangle over its own value, where that is not zero."""
    want = torch.triu(alpha * (x.double().t() @ x.double()))
    on = want != 0
    assert bool((got.double()[torch.triu(~on)] == 0).all())
    return float(((got.double() - want).abs()[on] / want.abs()[on]).max())


@pytest.mark.parametrize("left_out", PAIRS)
def test_bound_sees_each_product(left_out):
    x = _single_products(640, 770, 3)
    p = _planes(x)
    assert torch.equal(p[0] + p[1] + p[2], x.double())

    def total(pairs):
        return torch.triu(2 * sum(p[a].t() @ p[b] for a, b in pairs))

    assert _error(total(PAIRS), x) <= 1.01 * ULP
    assert _error(total([q for q in PAIRS if q != left_out]), x) > 4 * ONE_PRODUCT


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
@pytest.mark.parametrize("n,d", [(512, 512), (640, 770), (2049, 1001), (4096, 1024)])
def test_single_products(dev, n, d):
    x = _single_products(n, d, n + d)
    err = _error(_hessian(x.to(dev)).cpu(), x)
    print(f"single products {n} x {d}: {err / ULP:.2f} ulp", flush=True)
    assert err <= ONE_PRODUCT


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


@pytest.mark.gpu
@pytest.mark.parametrize("low", [40, 80, 100, 104, 110, 115, 120, 125])
def test_tiny_values_keep_their_bits(dev, low):
    """Columns of about 2^-low beside columns that bring the products back to
    about 1: the same bound, whatever the exponent.  (Products of two tiny
    columns underflow in fp32 arithmetic too.)"""
    n, d = 640, 770
    tiny = torch.arange(d) % 2 == 0
    g = torch.Generator()
    g.manual_seed(low)
    up = min(low, 60)
    x = _single_products(n, d, low, torch.where(tiny, torch.tensor(2.0) ** -low, torch.tensor(2.0) ** (up - 2)))
    got = _hessian(x.to(dev)).cpu()
    want = torch.triu(2 * (x.double().t() @ x.double()))
    mixed = torch.triu(tiny.unsqueeze(0) != tiny.unsqueeze(1)) & (want != 0)
    assert int(mixed.sum()) > 1000
    err = float(((got.double() - want).abs()[mixed] / want.abs()[mixed]).max())
    print(f"tiny values 2^-{low}: {err / ULP:.2f} ulp", flush=True)
    assert err <= ONE_PRODUCT


@pytest.mark.gpu
@pytest.mark.parametrize("n,d", [(512, 512), (512, 4096), (512, 8192), (640, 2560), (2048, 2048), (4096, 1000),
                                 (8192, 512), (8192, 4096), (16384, 2048), (32768, 1024), (8192, 8192)])
def test_no_further_from_64_bits_than_the_fp32_product(dev, n, d):
    """Short, long, narrow and wide calls: one token split to eight.  Equal
    column sizes, so that thousands of diagonal sums' errors count alike and
    neither side's is a matter of luck (measured 0.1 .. 0.7 of the fp32 product's)."""
    g = torch.Generator(device=dev)
    g.manual_seed(n + d)
    x = torch.randn(n, d, generator=g, device=dev)
    xd = x.double()
    want = torch.triu(2 * (xd.t() @ xd))
    err = [float((torch.triu(H).double() - want).norm() / want.norm()) for H in (_hessian(x), _fp32_product(x))]
    print(f"{n} x {d}: planes {err[0]:.2e}, fp32 product {err[1]:.2e}", flush=True)
    assert err[0] <= err[1]


@pytest.mark.gpu
@pytest.mark.parametrize("n,d", [(1024, 512), (4096, 1000)])
def test_columns_of_every_size_on_the_planes(dev, n, d):
    """Columns from 2^-59 to 2^48 (below 2^54 with their largest values, above
    2^-110 with their smallest), each to its own precision: errors over the
    product of the two columns' norms, no larger than the fp32 product's."""
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    x = torch.randn(n, d, generator=g, device=dev) * torch.pow(2.0, torch.linspace(-59, 48, d, device=dev))
    assert float(x.abs().max()) < 2.0 ** 54 and float(x[x != 0].abs().min()) >= 2.0 ** -110
    norm = x.double().norm(dim=0)
    want = torch.triu(x.double().t() @ x.double())
    on = torch.triu(torch.outer(norm, norm) > 2.0 ** -80)      # above the fp32 underflow of the sums' last bits
    err = [float(((torch.triu(H).double() / 2 - want) / torch.outer(norm, norm))[on].norm())
           for H in (_hessian(x), _fp32_product(x))]
    print(f"columns of every size {n} x {d}: planes {err[0]:.2e}, fp32 product {err[1]:.2e}", flush=True)
    assert not torch.equal(torch.triu(_hessian(x)), torch.triu(_fp32_product(x)))     # the planes took it
    assert err[0] <= err[1]


@pytest.mark.gpu
def test_no_memory_for_the_planes(dev):
    """The planes' workspace not to be had: the fp32 product, which needs none."""
    torch.cuda.empty_cache()    # no cached block that the workspace would fit
    x = torch.randn(65536, 1024, device=dev)
    H = torch.zeros(1024, 1024, device=dev)
    want = _fp32_product(x)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(dev).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(dev) + (32 << 20)) / total, dev)
    try:
        ops.hessian_syrk_(H, x, alpha=2.0, beta=0.0)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
    assert torch.equal(H, want)


@pytest.mark.gpu
@pytest.mark.parametrize("inf_at", [None, 5, -5], ids=["finite", "inf_in_first", "inf_in_last"])
@pytest.mark.parametrize("beta", [0.0, 0.5, 1.0])
@pytest.mark.parametrize("n,d", [(22093, 8192), (22272, 8200)])
def test_several_calls_of_planes(dev, n, d, beta, inf_at):
    """Rows whose planes would pass 1 GiB go in several calls (here 21760 rows,
    then 333, or four whole chunks of 128): beta counts once, the planes, their
    flag and the slots are used again, and one call may take the planes while the
    other, whose rows hold an infinity, takes the fp32 product.  The bound is the fp32 product's own error, doubled for
    the other order of its sum; the rows of the shorter call alone are 0.03 of H."""
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    x = torch.randn(n, d, generator=g, device=dev)
    c = 77
    if inf_at is not None:
        x[inf_at, c] = float("inf")
    H0 = 100 * torch.randn(d, d, generator=g, device=dev)
    H = ops.hessian_syrk_(H0.clone(), x, alpha=2.0, beta=beta)
    P = _fp32_product(x, 2.0, H0.clone(), beta)
    assert torch.equal(torch.tril(H, -1), torch.tril(H0, -1))
    if inf_at is not None:
        # the column meets every other one once, so its entries are the same infinities
        assert torch.equal(H[c, c:], P[c, c:]) and torch.equal(H[:c, c], P[:c, c])
        assert bool(torch.isinf(H[c, c:]).all())
        x[:, c] = 0
        for h in (H, P, H0):
            h[c, :] = 0
            h[:, c] = 0
    want = torch.mm(x.t().double(), x.double()).mul_(2)
    want.add_(H0.double(), alpha=beta).triu_()
    err = [float((torch.triu(h).double() - want).norm() / want.norm()) for h in (H, P)]
    print(f"{n} x {d}, beta {beta}, infinity at {inf_at}: {err[0]:.2e}, fp32 product {err[1]:.2e}", flush=True)
    assert err[0] <= 2 * err[1]
