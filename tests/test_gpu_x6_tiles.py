"""Batched inverse factors at orders and batches that take each tile of the
split products: remainders in rows, columns and K, triangular and lower-only
operands, one stage of K and several, against the factor in 64 bits.

Bound: the Hessians of 4 d random rows have a condition number kappa below
((1 + 1/2) / (1 - 1/2))^2 = 9 (Marchenko-Pastur), and a Cholesky factor and
triangular inverse of order d in fp32 are off by less than d kappa 2^-24
relative to the largest element; a wrong tile is off by its elements, which
are 1e-2 of it.

That bound does not see a missing plane product.  The elements 128 and more
off the diagonal do, all of which come from such products: relative to their
norm an fp32 chain is off by 3.7e-7 .. 4.2e-7 (torch on the CPU, these
Hessians; OFF is 3.5 times that), and one without h l', l h' or m m' by 3.2e-6
and more (checked below, on the CPU)."""
import pytest
import torch

from llmcompressor_amd import ops

OFF = 1.5e-6
PAIRS = ((0, 0), (0, 1), (1, 0), (0, 2), (2, 0), (1, 1))


def _hessian(d, g, device):
    x = torch.randn(4 * d, d, generator=g, device=device)
    return 2 * x.t() @ x


def _factor(H):
    """The factor of H / samples, damped, in 64 bits."""
    h = H.double().cpu() / (4 * H.shape[0])
    h.diagonal().add_(0.01 * h.diagonal().mean())
    return h, torch.linalg.cholesky(torch.linalg.inv(h), upper=True)


def _off_diagonal(got, ref):
    on = torch.triu(torch.ones_like(ref, dtype=torch.bool), 128)
    return float((got.double().cpu() - ref)[on].norm() / ref[on].norm())


def _planes(v):
    v = v.float()
    h = v.bfloat16().float()
    m = (v - h).bfloat16().float()
    return h.double(), m.double(), (v - h - m).bfloat16().double()


def _chain(h, pairs, nb=128):
    """The same factor by blocks, the products between blocks summed (in 64
    bits) from the given plane products."""
    d = h.shape[0]

    def product(a, b):
        p, q = _planes(a), _planes(b)
        return sum(p[i] @ q[j] for i, j in pairs)

    f, low, x = torch.flip(h, (0, 1)), torch.zeros_like(h), torch.zeros_like(h)
    for k in range(0, d, nb):
        a, b = slice(k, k + nb), slice(k + nb, d)
        low[a, a] = torch.linalg.cholesky(f[a, a])
        x[a, a] = torch.linalg.inv(low[a, a])
        if k + nb < d:
            low[b, a] = f[b, a] @ x[a, a].t()
            f[b, b] -= product(low[b, a], low[b, a].t())
    w = nb
    while w < d:
        for k in range(0, d - w, 2 * w):
            a, b = slice(k, k + w), slice(k + w, min(k + 2 * w, d))
            x[b, a] = -product(x[b, b], product(low[b, a], x[a, a]))
        w *= 2
    return torch.flip(x, (0, 1))


@pytest.mark.parametrize("left_out", [None, (0, 2), (2, 0), (1, 1), (0, 1), (0, 0)])
@pytest.mark.parametrize("d", [260, 388, 644])
def test_off_diagonal_bound_sees_each_product(d, left_out):
    h, ref = _factor(_hessian(d, torch.Generator().manual_seed(d), "cpu"))
    err = _off_diagonal(_chain(h, [p for p in PAIRS if p != left_out]), ref)
    assert err <= OFF / 10 if left_out is None else err > 2 * OFF


@pytest.mark.gpu
@pytest.mark.parametrize("d,batch", [(260, 3), (388, 40), (644, 64), (772, 64), (1092, 5), (1284, 16), (1540, 2)])
def test_batched_inverse_factor_matches_64_bits(dev, d, batch):
    print(f"x6 tiles: {batch} inverse factors of order {d}", flush=True)
    g = torch.Generator(device=dev).manual_seed(d)
    H = torch.empty(batch, d, d, device=dev)
    for b in range(batch):
        H[b] = _hessian(d, g, dev)
    hinv, _, ok = ops.gptq_hinv_batched(H, None, torch.full((batch,), 4.0 * d), 0.01)
    assert bool(ok.all())
    for b in {0, 1, batch - 1}:
        _, ref = _factor(H[b])
        err = ((hinv[b].double().cpu() - ref).abs().max() / ref.abs().max()).item()
        off = _off_diagonal(hinv[b], ref)
        print(f"  {b}: {err:.2e}, off the diagonal {off:.2e}", flush=True)
        assert err <= 9 * d * 2.0 ** -24
        assert off <= OFF
