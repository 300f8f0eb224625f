"""Batched inverse factors at orders and batches that take each tile of the
split products: remainders in rows, columns and K, triangular and lower-only
operands, one stage of K and several, against the factor in 64 bits.

Bound: the Hessians of 4 d random rows have a condition number kappa below
((1 + 1/2) / (1 - 1/2))^2 = 9 (Marchenko-Pastur), and a Cholesky factor and
triangular inverse of order d in fp32 are off by less than d kappa 2^-24
relative to the largest element; a wrong tile is off by its elements, which
are 1e-2 of it."""
import pytest
import torch

from llmcompressor_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,batch", [(260, 3), (388, 40), (644, 64), (772, 64), (1092, 5), (1284, 16), (1540, 2)])
def test_batched_inverse_factor_matches_64_bits(dev, d, batch):
    print(f"x6 tiles: {batch} inverse factors of order {d}", flush=True)
    g = torch.Generator(device=dev).manual_seed(d)
    H = torch.empty(batch, d, d, device=dev)
    for b in range(batch):
        x = torch.randn(4 * d, d, generator=g, device=dev)
        H[b] = 2 * x.t() @ x
    hinv, _, ok = ops.gptq_hinv_batched(H, None, torch.full((batch,), 4.0 * d), 0.01)
    assert bool(ok.all())
    for b in {0, 1, batch - 1}:
        h = H[b].double().cpu() / (4 * d)
        h.diagonal().add_(0.01 * h.diagonal().mean())
        ref = torch.linalg.cholesky(torch.linalg.inv(h), upper=True)
        err = ((hinv[b].double().cpu() - ref).abs().max() / ref.abs().max()).item()
        print(f"  {b}: {err:.2e}", flush=True)
        assert err <= 9 * d * 2.0 ** -24
