"""Permuted weight loads and stores against plain indexing.

Rows up to 64 KiB of LDS words are staged and gathered from there in calls of
3 x 2^18 elements or more; wider ones and smaller calls gather straight from
memory.  Both are exact copies (bf16 rounding is one conversion
of values torch rounds the same way), so everything compares bit for bit.
"""
import pytest
import torch

from llmcompressor_amd import ops

pytestmark = pytest.mark.gpu

# (batch, rows, cols): one row; rows that do not fill a workgroup's share;
# widths off every vector size; the widest staged rows and the first past
# them (stores: 16384 columns to bf16, 13107 to fp32; fp32 loads 16384)
SHAPES = [(1, 1, 8), (1, 9, 130), (3, 17, 1001), (2, 5, 4096), (1, 3, 13107), (1, 3, 13108), (1, 2, 16384),
          (1, 2, 16388),
          # staged: rows that do not fill the last workgroup's share of one to
          # eight, widths off every vector size, the widest staged rows and the
          # first past them, and the two sides of the least size
          (1, 787, 1001), (1, 97, 8200), (3, 2051, 130), (5, 1031, 514), (1, 61, 13107), (1, 61, 13108),
          (1, 49, 16384), (1, 49, 16388), (1, 1031, 8192), (1, 767, 1024), (1, 768, 1024)]


@pytest.mark.parametrize("batch,rows,cols", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_load_permuted(dev, batch, rows, cols, dtype):
    g = torch.Generator(device=dev)
    g.manual_seed(cols + rows)
    # rows of a wider matrix, so the row stride is not the width
    w = torch.randn(batch, rows, cols + 8, generator=g, device=dev).to(dtype)[:, :, 3:3 + cols]
    perm = torch.stack([torch.randperm(cols, generator=g, device=dev) for _ in range(batch)])
    dead = (torch.rand(batch, cols, generator=g, device=dev) < 0.1).int()
    want = torch.gather(w.float(), 2, perm.unsqueeze(1).expand(-1, rows, -1))
    assert torch.equal(ops.gptq_load_weight_batched(w, perm), want)
    got = ops.gptq_load_weight_batched(w, perm, dead)
    assert torch.equal(got, want.masked_fill(dead.bool().unsqueeze(1), 0.0))
    w0 = w[0].contiguous()   # aligned rows: the 16-byte path where the width allows it
    assert torch.equal(ops.gptq_load_weight(w0, perm[0]), want[0])


@pytest.mark.parametrize("batch,rows,cols", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("codes", [True, False])
def test_store_permuted(dev, batch, rows, cols, dtype, codes):
    g = torch.Generator(device=dev)
    g.manual_seed(cols + rows + 1)
    w = torch.randn(batch, rows, cols, generator=g, device=dev)
    c = torch.randint(-128, 128, (batch, rows, cols), generator=g, device=dev, dtype=torch.int8) if codes else None
    inv = torch.stack([torch.randperm(cols, generator=g, device=dev) for _ in range(batch)])
    at = inv.unsqueeze(1).expand(-1, rows, -1)
    out, cout = ops.gptq_store_weight_batched(w, inv, dtype, c)
    assert torch.equal(out, torch.gather(w, 2, at).to(dtype))
    assert cout is None if c is None else torch.equal(cout, torch.gather(c, 2, at))
