"""Integer codes in whole aligned chunks equal the general kernel's (which a
view off the alignment takes), as do 4-bit words packed from them."""
import pytest
import torch

from llmcompressor_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("zero_points", [False, True], ids=["sym", "asym"])
@pytest.mark.parametrize("strategy,group", [("tensor", None), ("channel", None), ("group", 8), ("group", 40),
                                            ("group", 128)])
@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 40), (33, 640), (257, 1032)])
def test_vector_codes_equal_general(dev, rows, cols, strategy, group, zero_points, dtype):
    if group and group > cols:
        pytest.skip("one whole group at least")
    print(f"quantize vec {rows}x{cols} {strategy} {group} {zero_points} {dtype}", flush=True)
    g = torch.Generator().manual_seed(rows * cols)
    wide = torch.randn(rows, cols + 8, generator=g).to(dtype)
    wide[0, 1], wide[-1, cols] = float("inf"), float("nan")
    wide = wide.to(dev)
    off = wide[:, 1:cols + 1]
    assert off.data_ptr() % 16
    ns = {"tensor": (1,), "channel": (rows, 1), "group": (rows, -(-cols // (group or 1)))}[strategy]
    scale = (torch.rand(ns, generator=g) * 0.4 + 0.02).to(dtype).to(dev)
    zp = torch.randint(-8, 8, ns, generator=g).to(torch.int8).to(dev) if zero_points else None
    for bits in (4, 8):
        a = ops.quantize_int(off, scale, zp, strategy, bits, group)
        b = ops.quantize_int(off.clone(memory_format=torch.contiguous_format), scale, zp, strategy, bits, group)
        assert torch.equal(a, b)
    c4 = ops.quantize_int(off, scale, zp, strategy, 4, group)
    u = (c4.to(torch.int64) + 8).reshape(rows, cols // 8, 8)
    words = (u << (4 * torch.arange(8, device=dev))).sum(-1)
    words = torch.where(words >= 2 ** 31, words - 2 ** 32, words).to(torch.int32)
    assert torch.equal(ops.pack_int32(c4, 4), words)


@pytest.mark.parametrize("symmetric", [True, False], ids=["sym", "asym"])
@pytest.mark.parametrize("strategy,group,block", [("channel", None, None), ("group", 16, None), ("group", 24, None),
                                                  ("group", 128, None), ("block", None, [5, 48])])
def test_typed_statistics_and_qparams_equal_converted(dev, strategy, group, block, symmetric):
    """bf16 statistics and scales and int8 zero points straight from the
    kernels are the converted fp32 ones, and the codes from either agree."""
    g = torch.Generator().manual_seed(5)
    x = torch.randn(37, 384, generator=g).to(torch.bfloat16)
    x[1], x[2] = 0, x[2].abs()
    x = x.to(dev)
    print(f"typed qparams {strategy} {group} {block} {symmetric}", flush=True)
    mn, mx = ops.observe_minmax(x, strategy, group, block)
    tn, tx = ops.observe_minmax(x, strategy, group, block, dtype=torch.bfloat16)
    assert tn.dtype == torch.bfloat16 and torch.equal(tn.float(), mn) and torch.equal(tx.float(), mx)
    for st in (torch.bfloat16, torch.float32):
        s, z = ops.calculate_qparams(mn, mx, -8, 7, symmetric, st)
        ts, tz = ops.calculate_qparams(tn, tx, -8, 7, symmetric, st, out_dtype=torch.bfloat16, zp_dtype=torch.int8)
        assert torch.equal(ts, s.to(torch.bfloat16)) and torch.equal(tz, z.to(torch.int8))
        a = ops.quantize_int(x, ts, tz, strategy, 4, group, block_structure=block, div_dtype=torch.bfloat16)
        b = ops.quantize_int(x, ts.float(), tz.float(), strategy, 4, group, block_structure=block,
                             div_dtype=torch.bfloat16)
        assert torch.equal(a, b)
