"""16-bit Hessians with less workspace than queried: the calls that one token
split (or few) can take run with those, and what needs a workspace whatever the
splits is refused."""
import ctypes as C

import pytest
import torch

from llmcompressor_amd import _lib as L
from llmcompressor_amd import ops

pytestmark = pytest.mark.gpu


def _rows(dev, n, d):
    g = torch.Generator(device=dev)
    g.manual_seed(n + d)
    return torch.randn(n, d, generator=g, device=dev).bfloat16()


def _close(H, x):
    want = torch.triu(2 * (x.double().t() @ x.double()))
    # bf16 products are exact; the sums of n rows round in fp32, to 1e-6 of the norm
    assert float((torch.triu(H).double() - want).norm() / want.norm()) <= 2e-6


@pytest.mark.parametrize("n,d", [(1024, 384), (2048, 512), (2080, 1024), (3968, 2048)])
def test_short_calls_run_without_a_workspace(dev, n, d):
    lib = L.lib()
    assert lib.mi355q_hessian_syrk_workspace_size(n, d, L.BF16) > 0
    x = _rows(dev, n, d)
    H = torch.zeros(d, d, device=dev)
    L.check(lib.mi355q_hessian_syrk(x.data_ptr(), L.BF16, n, d, d, H.data_ptr(), d, C.c_float(2.0), C.c_float(0.0),
                                    None, 0, L.stream_of(x)))
    _close(H, x)


def test_fewer_splits_in_a_smaller_workspace(dev):
    """4096 x 1024: two splits (20 slots of 256 KiB) where eight are asked for."""
    lib, n, d = L.lib(), 4096, 1024
    x = _rows(dev, n, d)
    nbytes = 20 << 18
    assert lib.mi355q_hessian_syrk_workspace_size(n, d, L.BF16) > nbytes
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    H = torch.zeros(d, d, device=dev)
    args = (x.data_ptr(), L.BF16, n, d, d, H.data_ptr(), d, C.c_float(2.0), C.c_float(0.0), ws.data_ptr())
    L.check(lib.mi355q_hessian_syrk(*args, nbytes, L.stream_of(x)))
    _close(H, x)
    assert lib.mi355q_hessian_syrk(*args, nbytes - 1, L.stream_of(x)) == L.INVALID_ARGUMENT
    assert b"workspace too small" in lib.mi355q_last_error()


def test_short_segments_run_without_a_workspace(dev):
    lib, d = L.lib(), 1024
    x = _rows(dev, 2048, d)
    parts = [x[:1024], x[1024:1500], x[1500:]]
    ptrs = (C.c_void_p * 3)(*[p.data_ptr() for p in parts])
    rows = (C.c_int64 * 3)(*[p.shape[0] for p in parts])
    assert lib.mi355q_hessian_syrk_segments_workspace_size(rows, 3, d, L.BF16) > 0
    H = torch.zeros(d, d, device=dev)
    L.check(lib.mi355q_hessian_syrk_segments(ptrs, rows, 3, L.BF16, d, d, H.data_ptr(), d, C.c_float(2.0),
                                             C.c_float(0.0), None, 0, L.stream_of(x)))
    _close(H, x)


@pytest.mark.parametrize("n,d,tiles", [(1024, 512, 3 * 4), (2048, 512, 3 * 8), (4096, 768, 6 * 8), (3072, 1280, 15 * 8),
                                       (8192, 512, 3 * 8 * 4)])
def test_short_calls_keep_whole_tiles(dev, n, d, tiles):
    """Partial tiles of 256 x 256: those that the choice of the splits counts, not
    up to four times as many; tails are cut into parts from 8192 tokens on."""
    assert L.lib().mi355q_hessian_syrk_workspace_size(n, d, L.BF16) == tiles << 18


@pytest.mark.parametrize("n,d", [(2080, 512), (2304, 512), (2336, 768), (8191, 512), (8192, 512), (8224, 1280)])
def test_uneven_splits_and_parts(dev, n, d):
    """Stages that do not divide by the splits, and the two sides of the line."""
    x = _rows(dev, n, d)
    H0 = torch.randn(d, d, device=dev)
    H = ops.hessian_syrk_(H0.clone(), x, alpha=2.0, beta=0.5)
    assert torch.equal(torch.tril(H, -1), torch.tril(H0, -1))
    want = torch.triu(2 * (x.double().t() @ x.double()) + 0.5 * H0.double())
    assert float((torch.triu(H).double() - want).norm() / want.norm()) <= 2e-6
