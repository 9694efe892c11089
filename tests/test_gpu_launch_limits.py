"""Calls whose streaming or K-split grid would reach 2^32 threads, of which a launch
runs the remainder only, without an error: they run on the element-wise
quantizers and the general product, whose grids are capped or smaller. Each
result equals, bit for bit, the two halves of the same call, which fit."""
from __future__ import annotations

import pytest
import torch

from practice_cuda_amd.impls.hip_per_block import hip_per_block_bmm
from practice_cuda_amd.impls.hip_per_channel import hip_per_channel_bmm, hip_per_channel_quant
from practice_cuda_amd.registry import QuantResult

pytestmark = pytest.mark.gpu
E4M3 = torch.float8_e4m3fn


def _same(whole, part):
    return torch.equal(whole.view(torch.uint8), part.view(torch.uint8))


@pytest.mark.parametrize("cols", [3, 8])
def test_many_short_rows(dev, cols):
    """One wave per row: 2^26 rows are 2^32 threads (odd rows, and rows of one aligned chunk)."""
    rows = 2 ** 26 + 5
    x = torch.randn(rows, cols, dtype=torch.bfloat16, device=dev)
    print(f"limits: {rows} rows of {cols}", flush=True)
    r = hip_per_channel_quant(x, channel_axis=-2)
    h = rows // 2
    for s in (slice(0, h), slice(h, rows)):
        p = hip_per_channel_quant(x[s], channel_axis=-2)
        assert _same(r.tensor[s], p.tensor) and _same(r.dequant_scale[s], p.dequant_scale)


def test_many_odd_columns(dev):
    """256 threads per 128 columns: 2^31 columns are 2^32 threads."""
    cols = 2 ** 31 + 5
    x = torch.randn(1, 2 ** 20 + 1, dtype=torch.bfloat16, device=dev).repeat(1, 2048)[:, :cols]
    x = x if x.shape[1] == cols else torch.nn.functional.pad(x, (0, cols - x.shape[1]), value=0.5)
    print(f"limits: {cols} columns", flush=True)
    r = hip_per_channel_quant(x, channel_axis=-1)
    h = 2 ** 30 + 1
    for s in (slice(0, h), slice(h, cols)):
        p = hip_per_channel_quant(x[:, s], channel_axis=-1)
        assert _same(r.tensor[:, s], p.tensor) and _same(r.dequant_scale[s], p.dequant_scale)


@pytest.mark.parametrize("scheme", ["channel", "block"])
def test_many_small_unaligned_products(dev, scheme):
    """2^23 products of one K-split tile of 512 threads (channel), or of two of 256 threads (block). The
    general kernel takes 256 threads for each."""
    batch = 2 ** 23 + 3
    m, n, k = (1, 1, 17) if scheme == "channel" else (17, 65, 17)
    g = torch.Generator(device=dev).manual_seed(1)
    a = torch.randint(-4, 5, (batch, m, k), generator=g, device=dev, dtype=torch.int8).to(torch.bfloat16).to(E4M3)
    b = torch.randint(-4, 5, (1, k, n), generator=g, device=dev, dtype=torch.int8).to(torch.bfloat16).to(E4M3)
    b = b.expand(batch, k, n)
    print(f"limits: {batch} products {scheme}", flush=True)
    if scheme == "channel":
        ra = QuantResult(a, torch.ones(batch, m, device=dev), "t", "channel", {"channel_axis": -2})
        rb = QuantResult(b, torch.ones(batch, n, device=dev), "t", "channel", {"channel_axis": -1})
        fn = hip_per_channel_bmm
    else:
        ra = QuantResult(a, torch.ones(batch, m, 1, device=dev), "t", "block", {"block_m": 1, "block_n": 128})
        rb = QuantResult(b, torch.ones(batch, 1, 1, device=dev), "t", "block", {"block_m": 128, "block_n": 128})
        fn = hip_per_block_bmm
    out = fn(ra, rb, out_dtype=torch.bfloat16)
    h = batch // 2
    for s in (slice(0, h), slice(h, batch)):
        half = [QuantResult(r.tensor[s], r.dequant_scale[s], "t", r.granularity, r.meta) for r in (ra, rb)]
        assert torch.equal(out[s], fn(*half, out_dtype=torch.bfloat16))
